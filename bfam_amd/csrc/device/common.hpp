/*
 * Device-side data layout shared by the stage, plain and reduction kernels.
 *
 * HBM layout of one volume subdomain (K elements, order N, Np nodes, NF
 * fields): element-major, field-major inside the element,
 *     q[e][f][n]   (state, two ping-pong copies for the fused stage)
 *     dq[e][f][n]  (LSRK rate register)
 * so a workgroup streams one contiguous NF*Np block per element and every
 * field row is a fully coalesced run of Np values.  Per-element geometry and
 * material live in small AoS tables (GEO_STRIDE / MAT_STRIDE entries), the
 * face connectivity in nbr_elem/nbr_code (one entry per element face).
 */
#pragma once

#include <hip/hip_runtime.h>
#include <stdint.h>

namespace bfamx
{

/* Pointers read out of a descriptor in memory are generic (flat) to the
 * compiler; casting them into the global address space lets loads and stores
 * use global_* instructions with a scalar base and a 32-bit lane offset
 * instead of 64-bit flat addresses per lane. */
template <class T>
using gptr = __attribute__((address_space(1))) T *;

template <class T> __device__ __forceinline__ gptr<T> glob(T *p)
{
  return (gptr<T>)(p);
}

/* Read-only tables that no kernel which reads them writes (task lists,
 * subdomain descriptors, clocks inside a stage launch, operators, element
 * material and connectivity) are read through the constant address space:
 * a wave-uniform load from it becomes a scalar load through the scalar data
 * cache, instead of a vector load queued behind the kernel's HBM streams
 * whose result must then be moved to a scalar register. */
template <class T>
using cptr = const __attribute__((address_space(4))) T *;

template <class T> __device__ __forceinline__ cptr<T> cglob(const T *p)
{
  return (cptr<T>)(p);
}

/* pointer to an element table: constant (scalar loads when the element is
 * uniform in the wave) or global address space */
template <bool SCALAR, class T> struct ElemPtr
{
  using type = gptr<const T>;
};
template <class T> struct ElemPtr<true, T>
{
  using type = cptr<T>;
};

enum
{
  GEO_GX = 0, /* 2/h_x, 2/h_y, 2/h_z : reference -> physical derivative */
  GEO_GY = 1,
  GEO_GZ = 2,
  GEO_LX = 3, /* lift factors (sJ/J)/w_end = (2/h_d)/w_0 */
  GEO_LY = 4,
  GEO_LZ = 5,
  GEO_X0 = 6, /* element lower corner */
  GEO_Y0 = 7,
  GEO_Z0 = 8,
  GEO_HX = 9,
  GEO_HY = 10,
  GEO_HZ = 11,
  GEO_STRIDE = 12
};

enum
{
  MAT_RHOI = 0, /* 1/rho */
  MAT_LAM = 1,  /* lambda (acoustic: bulk modulus) */
  MAT_MU = 2,
  MAT_ZP = 3, /* rho cp */
  MAT_ZS = 4, /* rho cs */
  MAT_STRIDE = 8
};

enum
{
  FMAT_ZP = 0,   /* plus-side rho cp */
  FMAT_ZS = 1,   /* plus-side rho cs */
  FMAT_IZP = 2,  /* 1 / (Zp- + Zp+) */
  FMAT_IZS = 3,  /* 1 / (Zs- + Zs+), 0 when both sides are fluid */
  FMAT_STRIDE = 4
};

enum
{
  MODE_STAGE = 0, /* RHS + LSRK update */
  MODE_RHS = 1    /* write L(q, t) as FP64 into rhs, no update */
};

/* parameters of one stage of a subdomain: 64 bytes, one scalar load.
 * parity: the stage reads q[parity] and writes q[parity ^ 1].
 * dq_dead: the dq this stage writes is never read (the last stage of a step
 *   of a scheme whose first stage has A = 0, every 2N-storage scheme here).
 *   Where dq is rebuilt from the states (rec), no stage stores it.
 * rec: B[s-1] times the old dq is q[parity] - q[parity ^ 1], and a holds
 *   A[s] / B[s-1].
 * g, sw, cw: ricker(t_stage), and sin, cos(omega t_stage) of the
 *   manufactured forcing. */
struct StageSlot
{
  int parity, dq_dead, rec, pad;
  double a, b, dt, g, sw, cw;
};

/* device-resident clock of one subdomain; all dynamic state lives here so a
 * captured graph can be replayed.  `ctx` holds the parameters of the next
 * CLOCK_SLOTS stages, counted from `stage`; a launch names its slot, so a
 * run of up to CLOCK_SLOTS stages (eight steps of five stages) needs one
 * clock kernel after its last stage.  With a one-thread clock kernel after
 * every stage, that kernel took 2.6 us of the 8.3 us of a small stage
 * (16 x 16 acoustic, FP64) and 4.6 us beside stages of 55-400 us: a chain of
 * dependent reads and FP64 exp and sincos. */
constexpr int CLOCK_SLOTS = 40;
struct Clock
{
  double t;        /* time at the start of the current step */
  double dt;       /* step size */
  long long stage; /* stages completed since set_fields */
  long long pad[5];
  StageSlot ctx[CLOCK_SLOTS];
};

/* everything a stage needs about one subdomain (passed by value or read
 * from a device table in batched launches) */
struct SubDev
{
  int physics;
  int N;
  int K;
  int nf;
  int nstages;
  int src_elem; /* -1 none */
  int mms;      /* 1: manufactured forcing */
  /* 1: stage s >= 1 rebuilds the previous dq from the two state buffers,
   * dq_{s-1} = (q_s - q_{s-1}) / B_{s-1}, and dq is never stored (state and
   * rates of one type, A[0] = 0, B[0..S-2] nonzero) */
  int dq_rec;
  void *q[2];   /* state ping-pong (double or float) */
  void *dq;     /* rate register (double or float); NULL with dq_rec */
  double *rhs;  /* FP64 RHS (plain path and MODE_RHS) */
  const int32_t *nbr_elem;
  const uint8_t *nbr_code;
  const double *geo;
  const float *geo_f;
  const double *mat;
  const float *mat_f;
  /* per element face: Zp+, Zs+, 1/(Zp- + Zp+), 1/(Zs- + Zs+) (0 if no S) */
  const double *fmat;
  const float *fmat_f;
  const double *Dr; /* (N+1)^2 column-major */
  const float *Dr_f;
  const double *r; /* LGL nodes */
  const double *w; /* LGL weights */
  double wi0;      /* 1 / w_0: lift weight of a face node relative to 2/h */
  const double *src_wt;
  const float *src_wt_f;
  const double *mms_tab; /* K x 3 axes x {sin, cos} x (N+1): sin/cos(k x) */
  const float *mms_tab_f;
  Clock *clock;
  /* glued faces (nbr_code & NBR_GLUED): nbr_elem is the offset of the
   * face's 6 x (N+1)^2 block in this buffer (arithmetic type), written by
   * the mortar kernel before each stage: dv[3], dT[3] per face node */
  void *glue_buf;
  double A[8], B[8], C[9];
  double AB[8]; /* the stage kernels' A: A[s] / B[s-1] with dq_rec, else A[s] */
  double src_amp[9];
  double src_f0, src_t0;
  double mms_k, mms_omega;
  double mms_F[9];
};

/* nbr_code flag of a face whose flux comes from the mortars */
constexpr int NBR_GLUED = 0x80;

/* nbr_code of a physical boundary face: NBR_BOUNDARY | kind << 3 | own face.
 * The plus state is the face's own trace, mirrored by kind:
 *   1 free surface (traction-free / pressure-free): v+ = v-, sigma+ = -sigma-
 *   2 rigid wall (no-slip / no normal flow):          v+ = -v-, sigma+ = sigma-
 *   3 absorbing (characteristic):                    v+ = 0,  sigma+ = 0
 * so that the exact Riemann solution at the face meets the condition. */
constexpr int NBR_BOUNDARY = 0x40;

/* orientation bits and mirror signs of a (non-glued) face code */
__device__ __forceinline__ int nbr_perm(int code)
{
  return (code & NBR_BOUNDARY) ? 0 : (code >> 3) & 7;
}
template <class T>
__device__ __forceinline__ void nbr_mirror(int code, T *sv, T *ss)
{
  if (!(code & NBR_BOUNDARY))
  {
    *sv = T(1);
    *ss = T(1);
    return;
  }
  const int kind = (code >> 3) & 7;
  *sv = kind == 1 ? T(1) : (kind == 2 ? T(-1) : T(0));
  *ss = kind == 1 ? T(-1) : (kind == 2 ? T(1) : T(0));
}

/* glued faces are at most order 7: (N+1)^2 <= 64 nodes, one per lane */
constexpr int GLUE_MAXFP = 64;

/* one interface handled by one wavefront of the mortar kernel: the b face
 * and its nm mortars (1: conforming, orders differ, quad0 = -1; 4: hanging,
 * mortar m is quadrant m of the b face).  *_off: offsets of the faces'
 * 6 x (N+1)^2 blocks in the glue buffer */
struct MortarGroup
{
  int32_t b_sub, b_elem, b_off;
  int32_t s_sub[4], s_elem[4], s_off[4];
  int8_t b_face, nm, quad0, pad;
  int8_t s_face[4];
  int8_t s_ng[4]; /* glue grid order of each mortar; 0: max(N_s, N_b) */
};

struct GlueArgs
{
  const SubDev *subs; /* the batch's descriptors */
  const MortarGroup *groups;
  int ngroups;
  int slot; /* as LaunchArgs::slot */
  const void *ops; /* glue_ops8_index table, arithmetic type */
  void *buf;       /* face fluctuation blocks */
};

/* 1-D mortar operators from order Na to Nb (1..8), column-major
 * (Nb+1) x (Na+1) in blocks of 81: kind 0 = prj[k], kind 1 = wi_mass_prj[k],
 * k = 0..4 as in create_interpolators */
__host__ __device__ constexpr int glue_ops_index(int kind, int Na, int Nb, int k)
{
  return ((((Na - 1) * 8 + (Nb - 1)) * 2 + kind) * 5 + k) * 81;
}
constexpr int GLUE_OPS_SIZE = 64 * 2 * 5 * 81;

/* the operators between orders 1..7 (the orders a face of the mortar
 * kernel can have), each padded to 8 x 8: entry (row, col) at row + 8 col,
 * zero outside the actual size; the mortar kernel's table */
__host__ __device__ constexpr int glue_ops8_index(int kind, int Na, int Nb, int k)
{
  return ((((Na - 1) * 7 + (Nb - 1)) * 2 + kind) * 5 + k) * 64;
}
constexpr int GLUE_OPS8_SIZE = 49 * 2 * 5 * 64;

/* one work item of a stage launch: elements [e0, e0+ne) of subdomain sub */
struct Task
{
  int sub;
  int e0;
  int ne;
  int N;
};

/* a value known to be the same in every lane, moved to a scalar register */
__device__ __forceinline__ float uniform(float v)
{
  return __builtin_bit_cast(float, __builtin_amdgcn_readfirstlane(__builtin_bit_cast(int, v)));
}
__device__ __forceinline__ double uniform(double v)
{
  const long long b = __builtin_bit_cast(long long, v);
  const int lo = __builtin_amdgcn_readfirstlane((int)(b & 0xffffffffLL));
  const int hi = __builtin_amdgcn_readfirstlane((int)(b >> 32));
  return __builtin_bit_cast(double, ((long long)hi << 32) | (unsigned int)lo);
}

/* field-wise load of a task from the global task table */
__device__ __forceinline__ Task load_task(const Task *tasks, int i)
{
  cptr<Task> t = cglob(tasks) + i;
  Task r;
  r.sub = t->sub;
  r.e0 = t->e0;
  r.ne = t->ne;
  r.N = t->N;
  return r;
}

struct LaunchArgs
{
  const SubDev *subs;       /* device table (batched) */
  const Task *tasks;        /* device table */
  int ntasks;
  int mode;
  int xcd_remap;
  int nxcd;
  /* stages launched since the clocks were last advanced: the stage's entry
   * of Clock::ctx */
  int slot;
  /* a launch over the whole of one subdomain, its tasks in element order:
   * the slots of its clock, its descriptor's index and its elements
   * (launch_task).  NULL: the task table and the descriptors' clocks. */
  const StageSlot *one;
  int one_sub, one_K;
  /* MODE_RHS: ricker(t), sin and cos(omega t) at the caller's time */
  double g_rhs, sw_rhs, cw_rhs;
};

/* Task i of a launch whose tasks hold TE elements.  ONE: computed where the
 * launch names its subdomain, and the stage parameters then loaded beside the
 * descriptor (stage_ctx): two dependent scalar loads fewer before a block
 * requests its state. */
template <int TE, bool ONE>
__device__ __forceinline__ Task launch_task(const LaunchArgs &a, int i)
{
  if (!ONE || !a.one)
    return load_task(a.tasks, i);
  const int e0 = i * TE, left = a.one_K - e0;
  return {a.one_sub, e0, left < TE ? left : TE, 0};
}

/* element-major offset of (element, field, node) */
__device__ __forceinline__ size_t qidx(int e, int f, int n, int NF, int Np)
{
  return ((size_t)e * NF + f) * Np + n;
}

/*
 * Order in which a block walks n tasks: task_at(v) for v = first, first +
 * stride, .. below end.  Hardware dispatches consecutive workgroups
 * round-robin over the XCDs.  Mode 0 keeps that order; mode 1 gives XCD x
 * the contiguous slice [x*C, (x+1)*C) of the (Morton-ordered) task list; mode
 * 2 (the default) keeps one round-robin front over the list but hands each
 * XCD whole Morton cubes of XC tasks, whose inner faces then share an L2.
 */
struct TaskWalk
{
  int first, stride, end;
};
__device__ __forceinline__ TaskWalk task_walk(const LaunchArgs &a, int n)
{
  const int b = blockIdx.x, G = gridDim.x;
  if (a.xcd_remap != 1 || G % a.nxcd)
    return {b, G, n};
  const int x = b % a.nxcd, s = b / a.nxcd, C = (n + a.nxcd - 1) / a.nxcd;
  const int lo = x * C, hi = lo + C;
  return {lo + s, G / a.nxcd, hi < n ? hi : n};
}
/* a grid whose blocks keep their XCD over the walk: every task its own
 * block, or a multiple of the XCDs */
template <int XC = 8>
__device__ __forceinline__ int task_at(const LaunchArgs &a, int n, int v)
{
  if (a.xcd_remap != 2 || a.nxcd != 8 || ((int)gridDim.x < n && gridDim.x % 8))
    return v;
  /* the XC blocks of each XCD in a group of 8 XC take one cube; of the
   * partial last group, cubes of 8 as far as they go, then the identity */
  const int g0 = v & ~(8 * XC - 1);
  if (g0 + 8 * XC <= n)
    return g0 + XC * (v & 7) + ((v & (8 * XC - 1)) >> 3);
  const int g1 = v & ~63;
  if (g1 + 64 > n)
    return v;
  return g1 + 8 * (v & 7) + ((v & 63) >> 3);
}

/* Ricker wavelet (1 - 2a) exp(-a), a = (pi f0 (t - t0))^2 */
__device__ __forceinline__ double ricker(double f0, double t0, double t)
{
  const double x = 3.14159265358979323846 * f0 * (t - t0);
  const double a = x * x;
  return (1 - 2 * a) * exp(-a);
}

/* stage parameters of a task's subdomain */
struct StageCtx
{
  int parity, dq_dead, rec;
  double a, b, dt;
  cptr<StageSlot> slot;
};

/* SD: SubDev, possibly qualified with the constant address space.  The
 * clock is constant within a stage launch: only clock_advance_kernel, a
 * separate launch, writes it. */
template <bool ONE = false, class SD>
__device__ __forceinline__ StageCtx stage_ctx(const SD &sd, const LaunchArgs &a)
{
  StageCtx c;
  const StageSlot *own = ((const Clock *)sd.clock)->ctx;
  c.slot = cglob(ONE && a.one ? a.one : own) + a.slot;
  const bool stage = a.mode != MODE_RHS;
  c.parity = c.slot->parity;
  c.dq_dead = stage ? c.slot->dq_dead : 0;
  c.rec = stage ? c.slot->rec : 0;
  c.a = stage ? c.slot->a : 0.0;
  c.b = stage ? c.slot->b : 0.0;
  c.dt = stage ? c.slot->dt : 0.0;
  return c;
}

/* the source and forcing scalars, loaded only where a task needs them: held
 * from the start of a task they cost the stage kernels registers */
__device__ __forceinline__ double stage_g(const StageCtx &c, const LaunchArgs &a)
{
  return a.mode == MODE_RHS ? a.g_rhs : c.slot->g;
}
__device__ __forceinline__ double stage_sw(const StageCtx &c, const LaunchArgs &a)
{
  return a.mode == MODE_RHS ? a.sw_rhs : c.slot->sw;
}
__device__ __forceinline__ double stage_cw(const StageCtx &c, const LaunchArgs &a)
{
  return a.mode == MODE_RHS ? a.cw_rhs : c.slot->cw;
}

/* the neighbour's node facing node nm of face f (non-glued faces): the
 * upload admits only axis-aligned connectivity, a neighbour meeting face f
 * with its opposite face f ^ 1 and unpermuted nodes, and boundary faces,
 * whose plus trace is the face's own */
__device__ __forceinline__ int nbr_node(int code, int f, int n1, int nm)
{
  if (code & NBR_BOUNDARY)
    return nm;
  const int stride = f < 2 ? 1 : (f < 4 ? n1 : n1 * n1);
  return (f & 1) ? nm - (n1 - 1) * stride : nm + (n1 - 1) * stride;
}

/* face permutation (swap / reverse bits), same as bfamx_perm_apply */
__device__ __forceinline__ int perm_apply(int code, int n1, int a, int b)
{
  int x = (code & 4) ? b : a;
  int y = (code & 4) ? a : b;
  if (code & 1)
    x = n1 - 1 - x;
  if (code & 2)
    y = n1 - 1 - y;
  return x + y * n1;
}

/* volume node of face f, in-face indices (a, b) (bfam.c:6599-6781 order) */
template <int DIM>
__device__ __forceinline__ int face_node(int f, int n1, int a, int b)
{
  const int fixed = (f & 1) ? n1 - 1 : 0;
  if (DIM == 2)
    return (f < 2) ? fixed + n1 * a : a + n1 * fixed;
  switch (f >> 1)
  {
  case 0: return fixed + n1 * (a + n1 * b);
  case 1: return a + n1 * (fixed + n1 * b);
  default: return a + n1 * (b + n1 * fixed);
  }
}

} // namespace bfamx
