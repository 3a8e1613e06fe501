/*
 * Field transfer between two adapted meshes (h-refine, h-coarsen, order
 * change), run once between steps after the mesh changes.
 *
 * The reference supplies the transfer maps (bfam_domain_pxest_transfer_
 * maps_init, bfam.c:5205-5387) and uploads, per order pair, the 1-D
 * operators Pr, Pr_cfb, Pr_cft, Pr_r2b, Pr_r2t (bfam.c:8399-8404, from
 * create_interpolators, bfam.c:5606); the kernel that applies them was
 * application code.  Here one workgroup builds one destination element:
 * three fields at a time and for each of its sources (one, or the eight
 * children of a coarsened element), the source element's values pass through
 * LDS three times, one 1-D operator along x, then y, then z (sum
 * factorisation: (N_d+1)(N_s+1)^3 + (N_d+1)^2 (N_s+1)^2 + (N_d+1)^3 (N_s+1)
 * multiply-adds instead of (N_d+1)^3 (N_s+1)^3), and the result adds into
 * accumulators that a thread keeps for its values of the destination.
 * Arithmetic is FP64 whatever the state types; each destination value is
 * rounded once to its state type.  A block is a chain of barriers, so what
 * counts is how few there are and how many blocks share a CU: three fields
 * take a third of the barriers of one, and without an accumulator in LDS six
 * blocks fit (5874 elements of orders 5 and 3, FP32: 273 -> 94 us with the
 * operators in LDS and the index divisions by multiplication).
 */
#include "launch.hpp"

namespace bfamx
{

constexpr int XFER_THREADS = 256;
constexpr int XFER_MAXNP = 512; /* (7+1)^3: elastic orders 3..7 */
constexpr int XFER_FIELDS = 3;  /* fields at a time */

template <class TS, class TD>
__global__ void __launch_bounds__(XFER_THREADS)
    transfer_kernel(const XferSide *__restrict__ srcs, const XferSide *__restrict__ dsts,
                    const XferTask *__restrict__ tasks, const double *__restrict__ ops)
{
  __shared__ double buf0[XFER_FIELDS * XFER_MAXNP], buf1[XFER_FIELDS * XFER_MAXNP];
  __shared__ double P[3][64];
  constexpr int R = XFER_FIELDS * XFER_MAXNP / XFER_THREADS;
  const int tid = threadIdx.x;
  cptr<XferTask> t = cglob(tasks) + blockIdx.x;
  cptr<XferSide> dd = cglob(dsts) + t->dst_sub;
  const int nsrc = t->nsrc, Nd = dd->N, nd = Nd + 1, npd = nd * nd * nd;
  /* n / nd = n md >> 16 exactly: md nd - 65536 < 8, and n < 8192 */
  const int md = (65535 + nd) / nd;
  gptr<TD> out = glob(static_cast<TD *>(dd->q)) + (size_t)t->dst_elem * 9 * npd;
  for (int f0 = 0; f0 < 9; f0 += XFER_FIELDS)
  {
    double acc[R];
#pragma unroll
    for (int r = 0; r < R; ++r)
      acc[r] = 0.0;
    for (int c = 0; c < nsrc; ++c)
    {
      cptr<XferSide> ss = cglob(srcs) + t->src_sub[c];
      const int Ns = ss->N, ns = Ns + 1, nps = ns * ns * ns, op = t->op[c];
      gptr<const TS> q = glob(static_cast<const TS *>(ss->q)) +
                         ((size_t)t->src_elem[c] * 9 + f0) * nps;
      __syncthreads(); /* buf0, P free (the previous z pass done) */
      for (int n = tid; n < XFER_FIELDS * nps; n += XFER_THREADS)
        buf0[n] = (double)q[n];
      if (f0 == 0 || nsrc > 1)
        if (tid < 3 * 64 && (tid & 63) < nd * ns)
          P[tid >> 6][tid & 63] =
              glob(ops)[glue_ops_index(0, Ns, Nd, (op >> (4 * (tid >> 6))) & 15) + (tid & 63)];
      __syncthreads();
      /* x: buf1[i + nd (j + ns (k + ns f))], i < nd, j, k < ns */
      for (int n = tid; n < XFER_FIELDS * nd * ns * ns; n += XFER_THREADS)
      {
        const int jkf = (n * md) >> 16, i = n - nd * jkf;
        double s = 0.0;
        for (int a = 0; a < ns; ++a)
          s += P[0][i + nd * a] * buf0[a + ns * jkf];
        buf1[n] = s;
      }
      __syncthreads();
      /* y: buf0[i + nd (j + nd (k + ns f))], i, j < nd, k < ns */
      for (int n = tid; n < XFER_FIELDS * nd * nd * ns; n += XFER_THREADS)
      {
        const int jkf = (n * md) >> 16, i = n - nd * jkf;
        const int kf = (jkf * md) >> 16, j = jkf - nd * kf;
        double s = 0.0;
        for (int a = 0; a < ns; ++a)
          s += P[1][j + nd * a] * buf1[i + nd * (a + ns * kf)];
        buf0[n] = s;
      }
      __syncthreads();
      /* z: value i + nd (j + nd (k + nd f)), i, j, k < nd */
#pragma unroll
      for (int r = 0; r < R; ++r)
      {
        const int n = tid + r * XFER_THREADS;
        if (n < XFER_FIELDS * npd)
        {
          const int jkf = (n * md) >> 16, kf = (jkf * md) >> 16, f = (kf * md) >> 16;
          const int ij = n - nd * nd * kf, k = kf - nd * f;
          double s = 0.0;
          for (int a = 0; a < ns; ++a)
            s += P[2][k + nd * a] * buf0[ij + nd * nd * (a + ns * f)];
          acc[r] += s;
        }
      }
    }
#pragma unroll
    for (int r = 0; r < R; ++r)
    {
      const int n = tid + r * XFER_THREADS;
      if (n < XFER_FIELDS * npd)
        out[f0 * npd + n] = (TD)acc[r];
    }
  }
}

hipError_t launch_transfer(int src_fp32, int dst_fp32, const XferSide *srcs,
                           const XferSide *dsts, const XferTask *tasks, int ntasks,
                           const double *ops, hipStream_t s)
{
  if (ntasks <= 0)
    return hipSuccess;
  const dim3 grid(ntasks), block(XFER_THREADS);
  if (src_fp32 && dst_fp32)
    transfer_kernel<float, float><<<grid, block, 0, s>>>(srcs, dsts, tasks, ops);
  else if (src_fp32)
    transfer_kernel<float, double><<<grid, block, 0, s>>>(srcs, dsts, tasks, ops);
  else if (dst_fp32)
    transfer_kernel<double, float><<<grid, block, 0, s>>>(srcs, dsts, tasks, ops);
  else
    transfer_kernel<double, double><<<grid, block, 0, s>>>(srcs, dsts, tasks, ops);
  return hipGetLastError();
}

} // namespace bfamx
