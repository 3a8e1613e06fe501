/*
 * Fused LSRK stage for 2-D velocity-pressure acoustics on affine
 * quadrilaterals (fields p, u, v):
 *   p_t = -K (u_x + v_y),  rho u_t = -p_x,  rho v_t = -p_y,  K = rho c^2.
 * Same structure as the elastic stage (see stage_elastic.hip); the upwind
 * fluctuation is the mu = 0 case of the elastic Riemann solution:
 *   dvn = (Z+ (vn+ - vn-) + (p- - p+)) / (Z- + Z+)
 *   rate_u += lift Z- dvn n / rho,   rate_p -= lift K dvn
 * (Hesthaven & Warburton 2008, sec. 2.4 upwind flux for linear systems).
 */
#include "physics.hpp"

namespace bfamx
{

template <int N, int EPB, class T> struct AcousticSmem
{
  static constexpr int n1 = N + 1, Np = n1 * n1;
  static constexpr int QW = EPB * 3 * Np;
  static constexpr int FW = EPB * 4 * n1;
  /* LDS: fields, face values, D */
  static constexpr size_t bytes = sizeof(T) * (QW + FW + n1 * n1);
};

template <int N, int EPB, class P, int PART = PART_FUSED, class SD>
__device__ __forceinline__ void acoustic_task(const SD &sd, const Task &tk,
                                              const StageCtx &cx, const LaunchArgs &la,
                                              char *smem)
{
  using TS = typename P::TS;
  using TR = typename P::TR;
  using TC = typename P::TC;
  constexpr int n1 = N + 1, Np = n1 * n1, Nfp = n1, NF = 3;
  constexpr int BS = EPB * Np;
  constexpr int NT = EPB * 4 * Nfp;
  constexpr int TPT = (NT + BS - 1) / BS;
  using SM = AcousticSmem<N, EPB, TC>;

  const int tid = threadIdx.x;
  const int le = tid / Np, n = tid - (tid / Np) * Np;
  const bool act = tid < BS && le < tk.ne;
  const int e = tk.e0 + le;
  const int i = n % n1, j = n / n1;

  TC *sq = reinterpret_cast<TC *>(smem); /* [EPB][3][Np] */
  TC *sfl = sq + SM::QW;                 /* [EPB][4][Nfp] */
  TC *sD = sfl + SM::FW;

  /* Everything the block reads from memory is requested here, the face traces
   * once the indices are there, so that a stage takes two round trips after
   * its descriptor's instead of five: a small subdomain's stage is that chain
   * of latencies, and a large one's occupancy covers them better.  us per
   * stage, loads at their use / here: FP64 N = 4 5.01 / 4.28 (16^2), 39.7 / 27.5
   * (256^2), N = 7 25.4 / 18.1 (128^2), FP32 N = 3 14.8 / 11.9 (256^2) */
  gptr<const TS> qin = glob(static_cast<const TS *>(sd.q[cx.parity]));
  int32_t ep[TPT];
  int code[TPT];
  if constexpr (PART != PART_VOLUME)
  {
#pragma unroll
    for (int r = 0; r < TPT; ++r)
    {
      const int t = tid + r * BS;
      const int lt = t / (4 * Nfp);
      if (tid < BS && t < NT && lt < tk.ne)
      {
        const size_t fi = (size_t)(tk.e0 + lt) * 4 + (t - lt * 4 * Nfp) / Nfp;
        ep[r] = glob(sd.nbr_elem)[fi];
        code[r] = glob(sd.nbr_code)[fi];
      }
    }
  }
  const bool upd = !(la.mode == MODE_RHS || PART != PART_FUSED);
  /* A = 0 (first stage of a step): no dq read.  FP32, FP64: the old dq is
   * rebuilt from the previous state, B_{s-1} dq_{s-1} = q_s - q_{s-1}, read
   * from the other ping-pong buffer before this thread overwrites the node (a
   * holds A_s / B_{s-1}) */
  const bool rd_dq = upd && cx.a != 0.0;
  constexpr bool REC = sizeof(TS) == sizeof(TR);
  const bool rec = REC && cx.rec;
  gptr<TS> qout = glob(static_cast<TS *>(sd.q[cx.parity ^ 1]));
  gptr<TR> dqp = glob(static_cast<TR *>(sd.dq));
  TS qs[NF];
  TR old[NF];
  TC rhoi = 0, bulk = 0, Zm = 0, gx = 0, gy = 0, lx = 0, ly = 0;
  if (act)
  {
#pragma unroll
    for (int f = 0; f < NF; ++f)
      qs[f] = qin[qidx(e, f, n, NF, Np)];
    gptr<const TC> M = mat_tab<TC>(sd) + (size_t)e * MAT_STRIDE;
    rhoi = M[MAT_RHOI];
    bulk = M[MAT_LAM];
    Zm = M[MAT_ZP];
    gptr<const TC> G = geo_tab<TC>(sd) + (size_t)e * GEO_STRIDE;
    gx = G[GEO_GX];
    gy = G[GEO_GY];
    lx = G[GEO_LX];
    ly = G[GEO_LY];
    if (rd_dq)
    {
      gptr<const TR> o = rec ? (gptr<const TR>)qout : (gptr<const TR>)dqp;
#pragma unroll
      for (int f = 0; f < NF; ++f)
        old[f] = o[qidx(e, f, n, NF, Np)];
    }
  }
  TC Dv = 0;
  gptr<const TC> Dg = dr_tab<TC>(sd);
  if (tid < n1 * n1)
    Dv = Dg[tid];
  /* plus trace (p, v_axis) and both impedances of this thread's face nodes */
  TS gp[TPT], gv[TPT];
  TC zm[TPT], zp[TPT];
  if constexpr (PART != PART_VOLUME)
  {
#pragma unroll
    for (int r = 0; r < TPT; ++r)
    {
      const int t = tid + r * BS;
      const int lt = t / (4 * Nfp);
      if (tid < BS && t < NT && lt < tk.ne)
      {
        const int rem = t - lt * 4 * Nfp;
        const int f = rem / Nfp, a = rem - (rem / Nfp) * Nfp;
        const int np = nbr_node(code[r], f, n1, face_node<2>(f, n1, a, 0));
        gp[r] = qin[qidx(ep[r], 0, np, NF, Np)];
        gv[r] = qin[qidx(ep[r], 1 + (f >> 1), np, NF, Np)];
        zm[r] = (mat_tab<TC>(sd) + (size_t)(tk.e0 + lt) * MAT_STRIDE)[MAT_ZP];
        zp[r] = (mat_tab<TC>(sd) + (size_t)ep[r] * MAT_STRIDE)[MAT_ZP];
      }
    }
  }
  if (tid < n1 * n1)
    sD[tid] = Dv;
  static_assert(BS >= n1 * n1, "one D entry per thread");
  if (act)
  {
#pragma unroll
    for (int f = 0; f < NF; ++f)
      sq[(le * NF + f) * Np + n] = (TC)qs[f];
  }
  __syncthreads();

  TC rate[NF];
  if (act && PART == PART_SURFACE)
  {
#pragma unroll
    for (int f = 0; f < NF; ++f)
      rate[f] = (TC)glob(sd.rhs)[qidx(e, f, n, NF, Np)];
  }
  if (act && PART != PART_SURFACE)
  {
    const TC *u = sq + le * NF * Np;
    TC px = 0, ux = 0, py = 0, vy = 0;
#pragma unroll
    for (int m = 0; m < n1; ++m)
    {
      const TC c = sD[i + m * n1];
      const int id = m + n1 * j;
      px += c * u[0 * Np + id];
      ux += c * u[1 * Np + id];
    }
#pragma unroll
    for (int m = 0; m < n1; ++m)
    {
      const TC c = sD[j + m * n1];
      const int id = i + n1 * m;
      py += c * u[0 * Np + id];
      vy += c * u[2 * Np + id];
    }
    px *= gx, ux *= gx, py *= gy, vy *= gy;
    rate[0] = -bulk * (ux + vy);
    rate[1] = -px * rhoi;
    rate[2] = -py * rhoi;
  }

  if constexpr (PART != PART_VOLUME)
  {
#pragma unroll
    for (int r = 0; r < TPT; ++r)
    {
      const int t = tid + r * BS;
      const int lt = t / (4 * Nfp);
      if (tid < BS && t < NT && lt < tk.ne)
      {
        const int rem = t - lt * 4 * Nfp;
        const int f = rem / Nfp, a = rem - (rem / Nfp) * Nfp;
        const int nm = face_node<2>(f, n1, a, 0);
        const TC *u = sq + lt * NF * Np;
        const TC s = (f & 1) ? TC(1) : TC(-1);
        TC sv, ss; /* pressure plays the stress: free surface p+ = -p- */
        nbr_mirror<TC>(code[r], &sv, &ss);
        const TC pm = u[nm], vnm = s * u[(1 + (f >> 1)) * Np + nm];
        const TC pp = ss * (TC)gp[r];
        const TC vnp = sv * s * (TC)gv[r];
        sfl[t] = (zp[r] * (vnp - vnm) + (pm - pp)) / (zm[r] + zp[r]);
      }
    }
    __syncthreads();

    if (act)
    {
      const TC *F = sfl + le * 4 * Nfp;
#define BFAMX_ALIFT(face, cond, fn_)                                           \
  if (cond)                                                                    \
  {                                                                            \
    const TC lift = (face) < 2 ? lx : ly;                                      \
    const TC dvn = F[(face)*Nfp + (fn_)];                                      \
    const TC sg = ((face)&1) ? TC(1) : TC(-1);                                 \
    rate[1 + ((face) >> 1)] += lift * Zm * dvn * sg * rhoi;                    \
    rate[0] -= lift * bulk * dvn;                                              \
  }
      BFAMX_ALIFT(0, i == 0, j)
      BFAMX_ALIFT(1, i == N, j)
      BFAMX_ALIFT(2, j == 0, i)
      BFAMX_ALIFT(3, j == N, i)
#undef BFAMX_ALIFT
    }
  }
  if (!act)
    return;

  if (PART != PART_SURFACE && e == sd.src_elem)
  {
    const TC g = (TC)stage_g(cx, la);
    const TC w = src_tab<TC>(sd)[n];
#pragma unroll
    for (int f = 0; f < NF; ++f)
      rate[f] += w * (TC)sd.src_amp[f] * g;
  }

  if (!upd)
  {
#pragma unroll
    for (int f = 0; f < NF; ++f)
      glob(sd.rhs)[qidx(e, f, n, NF, Np)] = (double)rate[f];
    return;
  }
  const TR ca = (TR)cx.a, cdt = (TR)cx.dt;
  const TS cb = (TS)cx.b;
#pragma unroll
  for (int f = 0; f < NF; ++f)
  {
    const size_t id = qidx(e, f, n, NF, Np);
    TR dqo = 0;
    if (rd_dq)
      dqo = rec ? (TR)qs[f] - old[f] : old[f];
    /* the product that is rounded by itself is named: left to contraction,
     * it is the one or the other by how the loads above compile, and an FP64
     * state under FP32 rates shows it (some 2e-8 of the state after 15 stages) */
    const TR d = fma(cdt, (TR)rate[f], ca * dqo);
    if (!cx.dq_dead && !rec)
      dqp[id] = d;
    qout[id] = qs[f] + cb * (TS)d;
  }
}

template <int N, int EPB, class P>
__global__ __launch_bounds__(EPB *(N + 1) * (N + 1)) void
acoustic_stage_kernel(LaunchArgs a)
{
  __shared__ __align__(16) char smem[AcousticSmem<N, EPB, typename P::TC>::bytes];
  const TaskWalk w = task_walk(a, a.ntasks);
  for (int v = w.first; v < w.end; v += w.stride)
  {
    const Task tk = launch_task<EPB, true>(a, task_at(a, a.ntasks, v));
    const auto &sd = *(cglob(a.subs) + tk.sub);
    const StageCtx cx = stage_ctx<true>(sd, a);
    acoustic_task<N, EPB, P>(sd, tk, cx, a, smem);
    __syncthreads();
  }
}

/* Blocks of up to 256 threads; for one subdomain (its tasks are then
 * computed) of at most SMALL_TASKS such tasks, blocks of as many elements as
 * one wavefront holds (N = 8: one element, 81 threads), which spreads it over
 * more CUs: few wavefronts then meet at each barrier.  Past some 128 tasks
 * the CUs are busy either way, and small blocks cost launches and repeated
 * loads of D.  us per stage, large / small blocks at about 32, 126 and 256
 * tasks: FP64 N = 2 4.92 / 4.55, 5.00 / 4.76, 5.09 / 5.26; N = 4 4.20 / 3.83,
 * 4.31 / 4.14, 4.40 / 4.60; N = 7 3.85 / 3.68, 3.90 / 3.77, 3.99 / 4.15; N = 8
 * 4.21 / 3.87, 4.29 / 4.23, 4.43 / 4.75; FP32 N = 4 4.16 / 3.76, 4.18 / 4.06,
 * 4.26 / 4.26; N = 8 3.99 / 3.75, 4.03 / 3.96, 4.09 / 4.17 */
constexpr int SMALL_TASKS = 128;

template <int N, class P>
static hipError_t launch_ae(const LaunchArgs &a, int grid, hipStream_t s)
{
  constexpr int Np = (N + 1) * (N + 1), E = 256 / Np, S = 64 / Np < 1 ? 1 : 64 / Np;
  if (a.one && a.ntasks <= SMALL_TASKS)
  {
    LaunchArgs b = a;
    b.ntasks = (a.one_K + S - 1) / S;
    const int nx = a.xcd_remap == 1 && a.nxcd > 1 ? a.nxcd : 1;
    hipLaunchKernelGGL((acoustic_stage_kernel<N, S, P>), dim3(nx * ((b.ntasks + nx - 1) / nx)),
                       dim3(S * Np), 0, s, b);
  }
  else
    hipLaunchKernelGGL((acoustic_stage_kernel<N, E, P>), dim3(grid), dim3(E * Np), 0, s, a);
  return hipGetLastError();
}

template <class P>
static hipError_t launch_an(int N, const LaunchArgs &a, int grid, hipStream_t s)
{
  switch (N)
  {
#define BFAMX_CASE(NN)                                                         \
  case NN: return launch_ae<NN, P>(a, grid, s);
    BFAMX_CASE(1)
    BFAMX_CASE(2)
    BFAMX_CASE(3)
    BFAMX_CASE(4)
    BFAMX_CASE(5)
    BFAMX_CASE(6)
    BFAMX_CASE(7)
    BFAMX_CASE(8)
#undef BFAMX_CASE
  default: return hipErrorInvalidValue;
  }
  return hipGetLastError();
}

hipError_t launch_acoustic_stage(int prec, int N, const LaunchArgs &a,
                                 int grid, hipStream_t s)
{
  switch (prec)
  {
  case PREC_FP32: return launch_an<P32>(N, a, grid, s);
  case PREC_FP32_RHS: return launch_an<P32R>(N, a, grid, s);
  default: return launch_an<P64>(N, a, grid, s);
  }
}

template <int N, int EPB, int PART>
__global__ __launch_bounds__(EPB *(N + 1) * (N + 1)) void
acoustic_part_kernel(LaunchArgs a)
{
  __shared__ __align__(16) char smem[AcousticSmem<N, EPB, double>::bytes];
  const TaskWalk w = task_walk(a, a.ntasks);
  for (int v = w.first; v < w.end; v += w.stride)
  {
    const Task tk = load_task(a.tasks, task_at(a, a.ntasks, v));
    const auto &sd = *(cglob(a.subs) + tk.sub);
    const StageCtx cx = stage_ctx(sd, a);
    acoustic_task<N, EPB, P64, PART>(sd, tk, cx, a, smem);
    __syncthreads();
  }
}

hipError_t launch_acoustic_plain(int N, const LaunchArgs &a, int grid,
                                 hipStream_t s)
{
  switch (N)
  {
#define BFAMX_CASE(NN)                                                         \
  case NN:                                                                     \
  {                                                                            \
    constexpr int E = 256 / ((NN + 1) * (NN + 1));                             \
    hipLaunchKernelGGL((acoustic_part_kernel<NN, E, PART_VOLUME>), dim3(grid), \
                       dim3(E * (NN + 1) * (NN + 1)), 0, s, a);                \
    hipLaunchKernelGGL((acoustic_part_kernel<NN, E, PART_SURFACE>),            \
                       dim3(grid), dim3(E * (NN + 1) * (NN + 1)), 0, s, a);    \
    break;                                                                     \
  }
    BFAMX_CASE(1)
    BFAMX_CASE(2)
    BFAMX_CASE(3)
    BFAMX_CASE(4)
    BFAMX_CASE(5)
    BFAMX_CASE(6)
    BFAMX_CASE(7)
    BFAMX_CASE(8)
#undef BFAMX_CASE
  default: return hipErrorInvalidValue;
  }
  return hipGetLastError();
}

} // namespace bfamx
