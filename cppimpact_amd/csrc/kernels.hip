// HIP kernels of the explicit-dynamics step for gfx950 and their launchers.
//
// One loop iteration of Dynamics::solve (dynamics.h:471-511) is, with the
// LDS-assembled scatter (the default):
//   k_elem_block4 (tet4; with the surrogate the elastic pass, k_mlp_queue
//                 and k_elem_block4_walk),
//   k_elem_block10 (tet10, 4-point rules), k_elem_block5 (tet10, 5 points)
//                 one workgroup per element block: stage the block's nodes
//                 in LDS, compute element forces (and the stress update),
//                 sum them per node in a fixed order, finish the nodes owned
//                 by the block (wall, gravity, leapfrog) and write one
//                 partial force per shared node
//   k_node_bnd    one thread per shared node: sum its partials in block
//                 order, then wall, gravity and leapfrog
// With the colour scatter k_elem_direct stores every corner force into the
// node's slot of the element's colour (no two elements of a colour share a
// node) and k_node_all sums a node's slots in colour order; with the atomic
// scatter it adds them with FP64 atomics, and k_node_all reads the sums.
//
// Nodal state: 24-byte records pos = x and vv = v, and the lumped mass m
// (read only by the nodes' owners: a step never writes it).
#include <hip/hip_ext.h>
#include <hip/hip_runtime.h>

#include <type_traits>

#include "device.h"
#include "elem.h"
#include "kernels.h"
#include "mlp_infer.h"

namespace cpi {

// ---------------------------------------------------------------------------
// reductions
// ---------------------------------------------------------------------------

// Sum / min over the wave, the same bits on every lane and in every run:
// each row of 16 lanes is reduced with DPP moves, then the four row values
// (lanes 0, 16, 32, 48) are combined in a fixed order.  All 64 lanes must
// be active.
__device__ __forceinline__ double wave_sum(double v) {
  v = row_reduce(v, [](double a, double b) { return a + b; });
  return (lane_value(v, 0) + lane_value(v, 16)) + (lane_value(v, 32) + lane_value(v, 48));
}
__device__ __forceinline__ double wave_min(double v) {
  v = row_reduce(v, [](double a, double b) { return fmin(a, b); });
  return fmin(fmin(lane_value(v, 0), lane_value(v, 16)), fmin(lane_value(v, 32), lane_value(v, 48)));
}

// wave_sum of a term that is zero on every lane of most waves (plastic
// work, inverted elements, penalty energy, contact force, and the nodal
// terms in the waves of an element kernel that update no node): a uniform
// branch skips the reduction then
__device__ __forceinline__ double wave_sum_sparse(double v) {
  return __ballot(v != 0.0) ? wave_sum(v) : 0.0;
}

// Each wave owns one energy row: its lanes' accumulators are reduced with
// wave_sum / wave_min (fixed order, so deterministic) and lane 0 updates the
// row; no workgroup barrier is involved.  Cumulative terms (internal and
// plastic work, gravity work, inverted-element count) accumulate in the row
// every step; the instantaneous ones (kinetic and penalty energy, contact
// force, stable dt) are only reduced on the steps that end a batch, the only
// ones whose rows are summed.  The row of a wave is base + its wave index in
// the grid.  The cumulative terms of the row are read when the kernel starts
// (row_prefetch), so the flush at its end only writes.
struct RowPre {
  double wint, wpl, bad, wgrav;
};

__device__ __forceinline__ RowPre row_prefetch(const Params &p, int base) {
  // wave-uniform address: the values land in scalar registers
  const int row = __builtin_amdgcn_readfirstlane(base + (int)(threadIdx.x >> 6));
  const double *r = p.epart + (long)row * EP_N;
  return RowPre{r[EP_WINT], r[EP_WPL], r[EP_BAD], r[EP_WGRAV]};
}

// Variants of the step kernels: a plain step; one with outputs; and one with
// outputs of a context that takes resident steps, which is left out when it
// was queued behind a launch that gave up.  It costs 0.2 to 0.7 us of a step
// with outputs of 24 to 32 us, and is a variant of its own because the step of
// a mesh too large to be resident lost 1-2% (1.57M tet4, FP64: 102 -> 104 us).
enum : int { STEP_PLAIN = 0, STEP_OUT = 1, STEP_OUT_ASK = 2 };
template <int AUX> __device__ __forceinline__ bool left_out(const Params &p) {
  return AUX == STEP_OUT_ASK && (p.ctl->decision & 1u);
}

// Scalar loads issued at the kernel's start (the energy row, dt) must not
// sink: the compiler moves them down to their first use, past the loads of
// the node records, where the whole workgroup then waits for another round
// trip before its first barrier.  A use here, in the block that issues them,
// keeps them where they are written.
__device__ __forceinline__ void keep_here(double &v) { asm volatile("" : "+s"(v)); }
__device__ __forceinline__ void keep_here(RowPre &r) {
  keep_here(r.wint);
  keep_here(r.wpl);
  keep_here(r.bad);
  keep_here(r.wgrav);
}

// The kernel's Params (its first argument) read again from the argument
// segment: for the body of a loop, where arguments held from before it spill
// a hundred scalar registers.  at: set once with params_at(), and made unknown
// to the compiler on every pass so that the loads stay in the body.
typedef const __attribute__((address_space(4))) Params *ParamsAt;
__device__ __forceinline__ ParamsAt params_at() {
  return (ParamsAt)__builtin_amdgcn_kernarg_segment_ptr();
}
__device__ __forceinline__ Params params_again(ParamsAt &at, const Params &p) {
  asm volatile("" : "+s"(at));
#ifdef __HIP_DEVICE_COMPILE__
  (void)p;
  return *at;
#else
  return p;  // the host pass knows no copy out of that address space
#endif
}

// One wave's energy terms into its row: the cumulative ones added to what
// the row held (pre), and with ALL the instantaneous ones (kinetic,
// penalty, contact force, stable dt) stored.
template <bool ALL>
__device__ __forceinline__ void wave_flush(const Params &p, int base, const EAcc &ea,
                                           const RowPre &pre) {
  const double wint = wave_sum(ea.wint), wpl = wave_sum_sparse(ea.wpl),
               bad = wave_sum_sparse(ea.bad), wg = wave_sum_sparse(ea.wgrav);
  double ke = 0.0, pen = 0.0, fc = 0.0, md = 0.0;
  if (ALL) {
    ke = wave_sum_sparse(ea.ke);
    pen = wave_sum_sparse(ea.pen);
    fc = wave_sum_sparse(ea.fc);
    md = wave_min(ea.mindt);
  }
  if ((threadIdx.x & 63) == 0) {
    double *r = p.epart + (long)(base + (threadIdx.x >> 6)) * EP_N;
    r[EP_WINT] = pre.wint + wint;
    r[EP_WPL] = pre.wpl + wpl;
    r[EP_BAD] = pre.bad + bad;
    r[EP_WGRAV] = pre.wgrav + wg;
    if (ALL) {
      r[EP_MINDT] = md;
      r[EP_KE] = ke;
      r[EP_PEN] = pen;
      r[EP_FC] = fc;
    }
  }
}

// ---------------------------------------------------------------------------
// node update: a = -f/m + wall + g; x += du; v += dt a  (dynamics.h:497-503,
// wall.h:37-44, dynamics_kernels.h:150-168).  The wall sees x + du = x_{n+1}.
// A held node (fixed set, when enabled) has a = 0 and no contact; its
// velocity is zero from the start, so it stays where it is.
// ---------------------------------------------------------------------------
struct NodeStep {
  double x[3], v[3];    // x_{n+1}, v_{n+3/2}
  double a[3], du[3];
};

// minv = 1 / m; contact: the wall acts on the node
__device__ __forceinline__ void node_advance(const Params &p, bool held, bool contact,
                                             const double f[3], const double x[3],
                                             const double v[3], double m, double minv, double dt,
                                             NodeStep &s, EAcc &ea) {
#pragma unroll
  for (int c = 0; c < 3; c++) {
    s.du[c] = dt * v[c];
    s.a[c] = (m != 0.0) ? minv * (-f[c]) : 0.0;
  }
  if (contact) {
#pragma unroll
    for (int c = 0; c < 3; c++) {
      if (c == p.wall_dim) {
        double pos = x[c] + s.du[c];
        double d = (pos - p.wall_loc) * p.wall_normal;
        if (d < 0.0) {
          s.a[c] += -1 * minv * d * p.wall_nk;
          ea.pen += 0.5 * p.wall_k * d * d;
          ea.fc += -p.wall_k * d;
        }
      }
    }
  }
  double ke = 0.0, wg = 0.0;
#pragma unroll
  for (int c = 0; c < 3; c++) {
    s.a[c] = held ? 0.0 : s.a[c] + p.grav[c];
    s.v[c] = v[c] + dt * s.a[c];
    double vi = s.v[c] - 0.5 * dt * s.a[c];
    ke += vi * vi;
    wg += p.grav[c] * s.du[c];
    s.x[c] = x[c] + s.du[c];
  }
  ea.ke += 0.5 * m * ke;
  ea.wgrav += m * wg;
}

__device__ __forceinline__ bool node_held(const Params &p, int g) {
  return p.fixed_mask && p.fixed_mask[g];
}
__device__ __forceinline__ bool node_contact(const Params &p, int g, bool held) {
  return p.wall_on && !held && (!p.contact_mask || p.contact_mask[g]);
}

template <bool AUX>
__device__ __forceinline__ void node_update(const Params &p, int g, const double f[3],
                                            const double x[3], const double v[3], double m,
                                            double dt, EAcc &ea) {
  const bool held = node_held(p, g);
  NodeStep s;
  node_advance(p, held, node_contact(p, g, held), f, x, v, m, 1.0 / m, dt, s, ea);
  p.pos[g] = Vec3{s.x[0], s.x[1], s.x[2]};
  p.vv[g] = Vec3{s.v[0], s.v[1], s.v[2]};
  if (AUX) {
    p.acc[g] = Node4{s.a[0], s.a[1], s.a[2], 0.0};
    p.du[g] = Node4{s.du[0], s.du[1], s.du[2], 0.0};
    p.xprev[g] = Node4{x[0], x[1], x[2], m};
  }
}

// N consecutive corner forces of local node j, ranks k..k+N-1 (k a multiple
// of N, N of 4, or below 4 read one by one), added to s in rank order.  All N
// slots are read before the first add, so their LDS latencies overlap.
template <int N, typename R>
__device__ __forceinline__ void node_force_batch(const R *lf, const uint16_t *joff, int j, int k,
                                                 R s[3]) {
  unsigned o[N];
  if constexpr (N >= 4) {
    const uint2 *w = reinterpret_cast<const uint2 *>(joff + k);
#pragma unroll
    for (int i = 0; i < N / 4; i++) {
      const uint2 u = w[i];
      o[4 * i] = u.x & 0xffffu;
      o[4 * i + 1] = u.x >> 16;
      o[4 * i + 2] = u.y & 0xffffu;
      o[4 * i + 3] = u.y >> 16;
    }
  } else {
#pragma unroll
    for (int i = 0; i < N; i++) o[i] = joff[k + i];
  }
  R v[N][3];
#pragma unroll
  for (int i = 0; i < N; i++) {
    const R *q = lf + 3 * (int)(o[i] + (unsigned)j);
#pragma unroll
    for (int c = 0; c < 3; c++) v[i][c] = q[c];
  }
#pragma unroll
  for (int i = 0; i < N; i++)
#pragma unroll
    for (int c = 0; c < 3; c++) s[c] += v[i][c];
}

// A local node's force from its deg corner-force slots in the block's LDS
// (jagged-diagonal: the k-th at off[k] + j), summed in slot order in the
// element precision R: FP64 for FP64 elements, FP32 for FP32 ones, whose
// element forces carry FP32 rounding already (the nodal update that
// follows is FP64 either way).  Eight slots at a time, then four, two and
// one by the bits of deg: a remainder taken slot by slot costs two dependent
// LDS reads per slot, up to seven times over.  With the scalar loads kept at
// the kernel's start (keep_here) the 1.57M-tet4 step went from 48.5 to 46.4
// us (FP64) and from 33.1 to 32.1 us (FP32), the 1.2M-tet10 one from 157.0
// to 153.8 us (FP32; FP64 within noise).
template <typename R>
__device__ __forceinline__ void node_force_sum(const R *lf, const uint16_t *joff, int j, int deg,
                                               double f[3]) {
  R s[3] = {R(0), R(0), R(0)};
  int k = 0;
  for (; k + 8 <= deg; k += 8) node_force_batch<8, R>(lf, joff, j, k, s);
  if (deg & 4) {
    node_force_batch<4, R>(lf, joff, j, k, s);
    k += 4;
  }
  if (deg & 2) {
    node_force_batch<2, R>(lf, joff, j, k, s);
    k += 2;
  }
  if (deg & 1) node_force_batch<1, R>(lf, joff, j, k, s);
  f[0] = double(s[0]);
  f[1] = double(s[1]);
  f[2] = double(s[2]);
}

// One block's partial force on a shared node, stored in the element
// kernel's precision: FP64 records (24 B) for FP64 elements, FP32 ones
// (12 B) for FP32 elements, whose element forces carry FP32 rounding
// already.  The boundary-node kernel sums them in FP64.
template <typename R>
__device__ __forceinline__ void store_partial(const Params &p, int slot, const double f[3]) {
  if constexpr (std::is_same<R, float>::value)
    reinterpret_cast<Vec3f *>(p.partial)[slot] = Vec3f{float(f[0]), float(f[1]), float(f[2])};
  else
    p.partial[slot] = Vec3{f[0], f[1], f[2]};
}

// A workgroup's LDS node records, structure of arrays of ml doubles each:
// x, y, z, m, vx, vy, vz.  Lanes gathering random nodes read 8-byte words at
// an 8-byte stride, so the reads spread over the LDS banks (records of 64
// bytes put every node on one of four bank groups).
struct LNodes {
  double *d;
  int ml;
  __device__ __forceinline__ void stage(int j, const Vec3 &x, double m, const Vec3 &vv) const {
    d[j] = x.x;
    d[ml + j] = x.y;
    d[2 * ml + j] = x.z;
    d[3 * ml + j] = m;
    d[4 * ml + j] = vv.x;
    d[5 * ml + j] = vv.y;
    d[6 * ml + j] = vv.z;
  }
  __device__ __forceinline__ void get(int l, double x[3], double v[3]) const {
#pragma unroll
    for (int c = 0; c < 3; c++) {
      x[c] = d[c * ml + l];
      v[c] = d[(4 + c) * ml + l];
    }
  }
  __device__ __forceinline__ double mass(int l) const { return d[3 * ml + l]; }
};

// bytes of the LDS regions of the workgroup element kernels: node records,
// corner forces (jagged-diagonal slots), the slot offsets off[k]
__host__ __device__ constexpr int lds_round16(long n) { return (int)(((n + 15) / 16) * 16); }
__host__ __device__ constexpr int lds_node_bytes(int ml) { return lds_round16(56L * ml); }
__host__ __device__ constexpr int lds_force_bytes(int rsz, int npe, int max_el) {
  return lds_round16((long)rsz * 3 * npe * max_el);
}
__host__ __device__ constexpr int lds_off_bytes(int kmax) { return lds_round16(2L * (kmax + 1)); }
__host__ __device__ constexpr int lds_basis_bytes(int npe, int rsz, int points) {
  return npe == 10 && rsz == 8 && points == 4 ? 8 * Tet10Basis<RULE_EXACT4>::n : 0;
}

// One element on the 5-point tet10 rule by five lanes, lane q's point q:
// slot(k) is where its force at corner k goes.  The force is the chain
// f = w_q detJ_q g_q + f over the points in rule order, which every lane runs
// on the value of the lane before it: after four steps the last point's lane
// has it, with the bits of one thread going through the points.  FP64 takes
// tet10_point_kin's arithmetic (f_q = M G summed in the same order); FP32 keeps
// tet10_point's, whose bits the direct kernels share.
template <int RULE, typename R, int PHYS, bool DEFER, class At, class Get, class Slot>
__device__ __forceinline__ void tet10_five(const Params &p, const At &at, const Get &get,
                                           const Slot &slot, R *lf, double dt, int e, int q,
                                           PreState<R> &pre, EAcc &ea) {
  constexpr int NQ = Quad<RULE>::n;
  auto store = [&](int k, const R f[3]) {
    if (q == NQ - 1) {
      R *dst = lf + 3 * slot(k);
#pragma unroll
      for (int c = 0; c < 3; c++) dst[c] = f[c];
    }
  };
  if constexpr (sizeof(R) == 8) {
    auto put = [&](int k, const R fq[3]) {
      R f[3] = {fq[0], fq[1], fq[2]};
#pragma unroll
      for (int s = 1; s < NQ; s++)
#pragma unroll
        for (int c = 0; c < 3; c++) f[c] = fq[c] + dpp_mov<kDppBefore>(f[c]);
      store(k, f);
    };
    double Ji[9], Lv[9], M[9];
    const double detJ = tet10_point_kin<RULE, R, PHYS>(p, get, q, Ji, Lv, ea);
    tet10_point_stress<RULE, R, PHYS, false, DEFER>(p, at, dt, e, q, pre, Ji, detJ, Lv, M, ea);
    tet10_point_forces<RULE, R>(q, M, put);
  } else {
    auto put = [&](int k, const R g[3], R wd) {
      R f[3];
#pragma unroll
      for (int c = 0; c < 3; c++) f[c] = fma(wd, g[c], R(0));
#pragma unroll
      for (int s = 1; s < NQ; s++)
#pragma unroll
        for (int c = 0; c < 3; c++) f[c] = fma(wd, g[c], dpp_mov<kDppBefore>(f[c]));
      store(k, f);
    };
    tet10_point<RULE, R, PHYS, true, DEFER>(p, at, get, dt, e, q, put, ea, &pre);
    if constexpr (PHYS != PHYS_COMPAT)
      if (q == 0) tet10_stable_dt<R>(p, get, ea);
  }
}

// ---------------------------------------------------------------------------
// LDS-assembled element pass, tet10 on the 5-point rule: five lanes per
// element, one per point, twelve elements per wave (four lanes idle; see
// tet10_five).  VALU-bound for a full chip.  Against one thread per element
// looping over the points (128 threads): 13k elements FP64 compat 18.9 -> 9.4
// us, FP32 15.6 -> 9.3, FP64 EP 23.2 -> 10.9; 663k elements 214 -> 141, FP32
// 127 -> 114, FP64 EP 319 -> 230, FP32 EP 180 -> 154 us.
// LDS: node records (LNodes), corner forces [max_el*10][3] R in jagged-
// diagonal slots (local node j's k-th contribution at off[k] + j), off[k].
// ---------------------------------------------------------------------------
template <int RULE, typename R, int PHYS, int AUX, int NT, int WPE>
__global__ void __launch_bounds__(NT) __attribute__((amdgpu_waves_per_eu(WPE)))
k_elem_block5(Params p) {
  extern __shared__ double smem[];
  constexpr int NQ = Quad<RULE>::n, EW = 64 / NQ, EB = NT / 64 * EW;
  const int b = xcd_remap(blockIdx.x, gridDim.x);
  RowPre row = row_prefetch(p, p.epart_base + b * (NT / 64));
  const int32_t *mt = p.meta + 8 * b;
  const int es = mt[0], nel = mt[1];
  const int ml = p.ml;
  const int32_t *nid = p.nid_pad + (long)b * ml;
  const LNodes ln{smem, ml};
  R *lf = (R *)((char *)smem + lds_node_bytes(ml));
  uint16_t *joff = (uint16_t *)((char *)lf + lds_force_bytes(sizeof(R), 10, p.max_el));
  const double dt = p.ctl->dt;
  const bool leave = left_out<AUX>(p);
  const int lane = threadIdx.x & 63, q = lane % NQ, te = (threadIdx.x >> 6) * EW + lane / NQ;

  // a thread's element words, local ids and slots two per word (rows of 20
  // bytes), and its point's state: the first element's before the nodes are
  // waited for, and the first node's places in the assembly too
  uint32_t lw[5], pw[5];
  PreState<R> pre;
  auto ahead = [&](int t) {
    const long e = es + (t < nel ? t : nel - 1);
#pragma unroll
    for (int k = 0; k < 5; k++) {
      lw[k] = reinterpret_cast<const uint32_t *>(p.conn_local + 10L * e)[k];
      pw[k] = reinterpret_cast<const uint32_t *>(p.csr_pos + 10L * e)[k];
    }
    if constexpr (PHYS != PHYS_COMPAT)
      load_state<false, R>(state_block<R>(p, b, NQ * t + q), true, pre);
  };
  const long o = (long)b * ml;
  const int j0 = threadIdx.x < ml ? threadIdx.x : ml - 1;
  const int g0 = nid[j0], slot0 = p.slot_pad[o + j0], deg0 = p.deg_pad[o + j0];
  ahead(te);
  for (int j = threadIdx.x; j < ml; j += NT) {
    const int g = j == threadIdx.x ? g0 : nid[j];
    if (g >= 0) ln.stage(j, p.pos[g], p.m[g], p.vv[g]);
  }
  for (int k = threadIdx.x; k <= p.kmax; k += NT) joff[k] = p.off_pad[(long)b * (p.kmax + 1) + k];
  __syncthreads();
  if (leave) return;

  EAcc ea;
  for (int t = te; lane < NQ * EW && t < nel; t += EB) {
    const int e = es + t;
    if (t != te) ahead(t);
    const StateBlock<R> at = state_block<R>(p, b, NQ * t + q);
    auto half = [](const uint32_t w[5], int k) {
      return (int)((w[k >> 1] >> (16 * (k & 1))) & 0xffffu);
    };
    auto get = [&](int k, double xk[3], double vk[3]) { ln.get(half(lw, k), xk, vk); };
    auto slot = [&](int k) { return half(pw, k); };
    tet10_five<RULE, R, PHYS, false>(p, at, get, slot, lf, dt, e, q, pre, ea);
  }
  __syncthreads();

  for (int j = threadIdx.x; j < ml; j += NT) {
    const bool first = j == threadIdx.x;
    const int g = first ? g0 : nid[j];
    if (g < 0) continue;
    double f[3];
    node_force_sum<R>(lf, joff, j, first ? deg0 : p.deg_pad[o + j], f);
    const int slot = first ? slot0 : p.slot_pad[o + j];
    if (slot < 0) {
      double x[3], v[3];
      ln.get(j, x, v);
      node_update<AUX != 0>(p, g, f, x, v, ln.mass(j), dt, ea);
    } else {
      store_partial<R>(p, slot, f);
    }
  }
  wave_flush<AUX != 0>(p, p.epart_base + b * (NT / 64), ea, row);
}

// A workgroup's elements on a 4-point tet10 rule: the corner forces into the
// block's slots.  cw: the corner words of the thread's element e, of the
// block's last one in threads without (has_e false); some: the wave has an
// element.  Lane q stores corners q, q + 4 and q + 8.
template <int RULE, typename R, int PHYS, bool STREAM, bool DEFER, bool MM, class At>
__device__ __forceinline__ void tet10_block(const Params &p, const At &at, const LNodes &ln,
                                            R *lf, const uint16_t *joff, const double *basis,
                                            const uint32_t cw[5], double dt, int e, int t, int q,
                                            bool has_e, bool some, PreState<R> &pre, EAcc &ea) {
  auto half = [&](int k) { return (int)((cw[k >> 1] >> (16 * (k & 1))) & 0xffffu); };
  auto get = [&](int k, double x[3], double v[3]) { ln.get(half(k) & 511, x, v); };
  int sl[3];
#pragma unroll
  for (int j = 0; j < 3; j++) {
    const uint32_t lo = cw[2 * j], hi = cw[j == 2 ? 4 : 2 * j + 1];
    const int h = (int)(((q >> 1 ? hi : lo) >> (16 * (q & 1))) & 0xffffu);
    sl[j] = (int)joff[h >> 9] + (h & 511);
  }
  auto store = [&](int j, const R f[3]) {
    R *dst = lf + 3 * sl[j];
    dst[0] = f[0];
    dst[1] = f[1];
    dst[2] = f[2];
  };
  R Ji[9], Lv[9], M[9] = {};
  if (has_e) {
    const R detJ = tet10_point_kin<RULE, R, PHYS>(p, get, q, Ji, Lv, ea);
    tet10_point_stress<RULE, R, PHYS, STREAM, DEFER>(p, at, dt, e, q, pre, Ji, detJ, Lv, M, ea);
  }
  if constexpr (MM) {
    if (!__builtin_amdgcn_readfirstlane(some)) return;
    auto put = [&](int g, const double f[3]) {
      if (has_e && (g < 2 || q < 2)) store(g, f);
    };
    tet10_wave_forces(basis, t & 63, M, put);
  } else if (has_e) {
    auto put = [&](int k, const R fq[3]) {
      const R f[3] = {quad_sum(fq[0]), quad_sum(fq[1]), quad_sum(fq[2])};
      if ((k & 3) == q) store(k >> 2, f);
    };
    tet10_point_forces<RULE, R>(q, M, put);
  }
}

// tet10 on a 4-point rule: four lanes per element, one per quadrature point
// (PointLane), so a workgroup of NT threads holds at most NT/4 elements, and
// the plan gives it at most NT local nodes, one per thread.
// As in the tet4 kernel every global load of the workgroup (the node's id,
// slot and contribution count, the node records and slot offsets, the
// element's ten corner words, the point's stress state with its ep only
// when the point's yielded bit says it has yielded) is issued before the
// first barrier; after it the element pass reads only LDS and the node pass
// only LDS and its registers.  Lane q of an element stores corners q, q + 4
// and q + 8 (summed over the element's four points) into the corner's
// jagged-diagonal slot, off[rank] + local node; the nodes are then assembled
// as in k_elem_block5, and the point's state is stored last.  LDS as
// k_elem_block5, then the basis gradients (MM).
template <int RULE, typename R, int PHYS, int AUX, int NT, int WPE, bool STREAM, bool MM>
__global__ void __launch_bounds__(NT) __attribute__((amdgpu_waves_per_eu(WPE)))
k_elem_block10(Params p) {
  extern __shared__ double smem[];
  const int b = xcd_remap(blockIdx.x, gridDim.x);
  const int t = threadIdx.x;
  const PointLane<MM> pt(t);
  const int q = pt.q;
  RowPre row = row_prefetch(p, p.epart_base + b * (NT / 64));
  const int32_t *mt = p.meta + 8 * b;
  const int es = mt[0], nel = mt[1];
  const LNodes ln{smem, p.ml};
  R *lf = (R *)((char *)smem + lds_node_bytes(p.ml));
  uint16_t *joff = (uint16_t *)((char *)lf + lds_force_bytes(sizeof(R), 10, p.max_el));
  double *basis = (double *)((char *)joff + lds_off_bytes(p.kmax));
  double dt = p.ctl->dt;
  const bool leave = left_out<AUX>(p);
  // yielded bits, one per lane (point) of the wave: a point's ep is read
  // only when it has yielded before
  const int wv = __builtin_amdgcn_readfirstlane(t >> 6);
  const bool has_word = PHYS == PHYS_EP && p.yielded && wv < p.ywords;
  const long yi = (long)b * p.ywords + wv;
  unsigned long long yw = ~0ull;
  if (has_word) yw = p.yielded[yi];
  // the loads in the order of the tet4 body (block4): node ids, then the
  // node records and slot offsets, then corner words and stress state, with
  // no branch between them (one offset per thread: kmax <= max_el <= NT/4)
  const long o = (long)b * p.ml + (t < p.ml ? t : p.ml - 1);
  const int slot_o = p.slot_pad[o], deg_o = p.deg_pad[o], g_o = p.nid_pad[o];
  const bool has_n = t < p.ml && g_o >= 0;
  const int g = has_n ? g_o : -1, slot = has_n ? slot_o : -1, deg = has_n ? deg_o : 0;
  const Vec3 xr = p.pos[has_n ? g_o : 0];
  const double mr = p.m[has_n && slot_o < 0 ? g_o : 0];
  const Vec3 vr = p.vv[has_n ? g_o : 0];
  const uint16_t jo = p.off_pad[(long)b * (p.kmax + 1) + (t < p.kmax ? t : p.kmax)];
  [[maybe_unused]] double gk = 0.0;
  if constexpr (MM)
    gk = tet10_basis<RULE>.v[t < Tet10Basis<RULE>::n ? t : Tet10Basis<RULE>::n - 1];
  __builtin_amdgcn_sched_barrier(0);
  const bool has_e = pt.el < nel;
  const int e = es + pt.el, ec = has_e ? e : es + nel - 1;
  const StateBlock<R> at = state_block<R>(p, b, pt.place(p));
  // the element's ten corner words (local node | rank << 9), two per word
  // (the rows of 20 bytes are 4-byte aligned)
  uint32_t cw[5];
  {
    const uint32_t *cp = reinterpret_cast<const uint32_t *>(p.corner + 10L * ec);
#pragma unroll
    for (int k = 0; k < 5; k++) cw[k] = cp[k];
  }
  PreState<R> pre;
  if constexpr (PHYS != PHYS_COMPAT)
    load_state<STREAM, R>(at, (yw >> (t & 63)) & 1ull, pre);
  __builtin_amdgcn_sched_barrier(0);
  keep_here(dt);
  keep_here(row);
  if (has_n) ln.stage(t, xr, mr, vr);
  if (t <= p.kmax) joff[t] = jo;
  if constexpr (MM)
    if (t < Tet10Basis<RULE>::n) basis[t] = gk;
  __syncthreads();
  if (leave) return;

  EAcc ea;
  // set where the point is computed: a lane without one never reads its
  // loaded state again, so nothing after the element pass waits for the
  // state loads (nor, by the in-order wait count, for the state stores)
  bool yielded = false;
  tet10_block<RULE, R, PHYS, STREAM, !AUX, MM>(p, at, ln, lf, joff, basis, cw, dt, e, t, q, has_e,
                                               pt.el - (t & 15) < nel, pre, ea);
  if (has_e) yielded = pre.ep > R(0);
  if constexpr (PHYS == PHYS_EP) {
    const unsigned long long nb = __ballot(yielded);
    if (has_word && (t & 63) == 0 && nb != yw) p.yielded[yi] = nb;
  }
  __syncthreads();

  if (g >= 0) {
    double f[3];
    node_force_sum<R>(lf, joff, t, deg, f);
    if (slot < 0) {
      double x[3], v[3];
      ln.get(t, x, v);
      node_update<AUX != 0>(p, g, f, x, v, ln.mass(t), dt, ea);
    } else {
      store_partial<R>(p, slot, f);
    }
  }
  wave_flush<AUX != 0>(p, p.epart_base + b * (NT / 64), ea, row);
  // the point's state last (tet10_point_stress leaves it in pre), except in
  // the once-per-batch variant, whose outputs leave no registers for it
  if constexpr (PHYS != PHYS_COMPAT && !AUX)
    if (has_e) store_state<STREAM, R>(at, pre.s, pre.ep, pre.changed);
}

// tet4: the plan gives every workgroup at most NT elements and NT local
// nodes, so each thread owns one element and at most one node, and every
// global load of the workgroup (stress state, corner words, the
// contribution lists, node records, slots) is issued before the first
// barrier.  LDS: node records (LNodes), corner forces [max_el*4][3] R in
// jagged-diagonal slots, the slot offsets off[k].
//
// With the surrogate (PHYS_EP_MLP, FP32) a step is three launches:
//   elastic pass  this body over every block (WALK = false): a block whose
//                 trial stresses all stay inside the yield surface finishes
//                 here; a block with a yielding element writes nothing of
//                 its state, queues the network inputs of its yielding
//                 points (in thread order) and lists itself (one 64-bit
//                 atomic per deferred block: list slot and first queue row)
//   k_mlp_queue   the network on the whole queue (mlp_infer.h)
//   walk          this body (WALK = true) over the listed blocks: yielding
//                 elements take their queued outputs through mlp_apply
//                 (acceptance checks, FP64 exact fallback)
// A deferred block computes the same trial stresses, hence the same
// yielding set and queue order, in both launches, and which workgroup
// finishes a block never changes its results.
// CW: the element's corners as 16-bit words l | k << 9 (p.corner, 8 B per
// element), the slot off[k] + l taken from the LDS offsets after the
// barrier; otherwise the local ids and slots as two u16 arrays (16 B), for
// plans whose blocks exceed the words (a node in more than 128 elements of
// one block).
template <typename R, int PHYS, int AUX, int NT, bool WALK, bool STREAM, bool CW>
__device__ __forceinline__ void block4(const Params &p, const int b, const unsigned qbase,
                                       int *wcnt, unsigned *misc) {
  extern __shared__ double smem[];
  const int t = threadIdx.x, w = t >> 6, lane = t & 63;
  RowPre row = row_prefetch(p, p.epart_base + b * (NT / 64));
  const int32_t *mt = p.meta + 8 * b;
  const int es = mt[0], nel = mt[1];
  const LNodes ln{smem, p.ml};
  R *lf = (R *)((char *)smem + lds_node_bytes(p.ml));
  uint16_t *joff = (uint16_t *)((char *)lf + lds_force_bytes(sizeof(R), 4, p.max_el));
  double dt = p.ctl->dt;
  const bool leave = left_out<AUX>(p);
  // the FP64 EP body has no register to hold the answer in: it leaves at once
  constexpr bool kEarly = sizeof(R) == 8 && PHYS == PHYS_EP;
  if (kEarly && leave) return;

  // yielded bits of this wave's elements: a block has ywords words, one
  // per 64 elements of the largest block, and a wave past them (a block
  // plan of at most 320 elements per block) has no elements and no word
  const int wv = __builtin_amdgcn_readfirstlane(t >> 6);
  const bool has_word = PHYS != PHYS_COMPAT && p.yielded && wv < p.ywords;
  const long yi = (long)b * p.ywords + wv;
  unsigned long long yw = ~0ull;
  if (has_word) yw = p.yielded[yi];
  // The loads of the workgroup, issued with no branch between them in the
  // order they are needed: the node ids, slots and degrees (fixed stride,
  // the record addresses depend on them), then the node records and the
  // slot offsets the first barrier waits for, then the corner words and
  // the stress state, which stay in flight across the barrier until the
  // element pass uses them.  Lanes past the block's nodes or elements load
  // the last valid entry and drop it.  One offset per thread covers the
  // block: kmax (the largest contribution count) <= max_el <= NT.
  const long o = (long)b * p.ml + (t < p.ml ? t : p.ml - 1);
  const int slot_o = p.slot_pad[o], deg_o = p.deg_pad[o], g_o = p.nid_pad[o];
  const bool has_n = t < p.ml && g_o >= 0;
  const int g = has_n ? g_o : -1, slot = has_n ? slot_o : -1, deg = has_n ? deg_o : 0;
  const Vec3 xr = p.pos[has_n ? g_o : 0];
  const double mr = p.m[has_n && slot_o < 0 ? g_o : 0];
  const Vec3 vr = p.vv[has_n ? g_o : 0];
  const uint16_t jo = p.off_pad[(long)b * (p.kmax + 1) + (t < p.kmax ? t : p.kmax)];
  __builtin_amdgcn_sched_barrier(0);
  const bool has_e = t < nel;
  const int e = es + t, ec = has_e ? e : es + nel - 1;
  const StateBlock<R> at = state_block<R>(p, b, t);
  const uint2 lc4 = *(const uint2 *)((CW ? p.corner : p.conn_local) + 4L * ec);
  uint2 ps4 = make_uint2(0u, 0u);
  if constexpr (!CW) ps4 = *(const uint2 *)(p.csr_pos + 4L * ec);
  PreState<R> pre;
  if constexpr (PHYS != PHYS_COMPAT)
    load_state<STREAM, R>(at, (yw >> (t & 63)) & 1ull, pre);
  __builtin_amdgcn_sched_barrier(0);
  keep_here(dt);
  keep_here(row);
  if (has_n) ln.stage(t, xr, mr, vr);
  if (t <= p.kmax) joff[t] = jo;
  if constexpr (WALK)
    if (t == 0) misc[0] = misc[1] = 0u;
  __syncthreads();
  if (!kEarly && leave) return;

  EAcc ea;
  // corner k's 16-bit field of the two loaded words: its local id for the
  // gather and its slot for the force, decoded where they are used, or up
  // front in the walk (each form the one with fewer VGPRs)
  auto half = [&](const uint2 &u, int k) -> int {
    const unsigned v = k < 2 ? u.x : u.y;
    return (int)((k & 1) ? (v >> 16) : (v & 0xffffu));
  };
  auto lid = [&](int k) -> int { return CW ? (half(lc4, k) & 511) : half(lc4, k); };
  auto pos = [&](int k) -> int {
    const int h = half(lc4, k);
    return CW ? joff[h >> 9] + (h & 511) : half(ps4, k);
  };
  [[maybe_unused]] int l[4], ps[4];
  if constexpr (WALK) {
#pragma unroll
    for (int k = 0; k < 4; k++) {
      l[k] = lid(k);
      ps[k] = pos(k);
    }
  }
  auto get = [&](int k, double xk[3], double vk[3]) {
    if constexpr (WALK)
      ln.get(l[k], xk, vk);
    else
      ln.get(lid(k), xk, vk);
  };
  auto put = [&](int k, const R fk[3]) {
    R *dst;
    if constexpr (WALK)
      dst = lf + 3 * ps[k];
    else
      dst = lf + 3 * pos(k);
#pragma unroll
    for (int c = 0; c < 3; c++) dst[c] = fk[c];
  };
  [[maybe_unused]] R Ji[9], de[6], wd, snew[6], wk;
  [[maybe_unused]] bool yielding = false, ep_changed = false;
  // set where the element is computed (as in k_elem_block10)
  [[maybe_unused]] bool has_ep = false;
  if (has_e) {
    if constexpr (PHYS == PHYS_EP_MLP) {
      // an element whose trial stress stays inside the yield surface
      // finishes here; a yielding one waits for the network
      tet4_kin<R, PHYS_EP_MLP>(p, get, dt, Ji, de, wd, ea);
      wk = ep_trial<R>(p, de, pre.s, snew);
      if (!trial_yields<R>(p, snew, pre.ep)) {
#pragma unroll
        for (int c = 0; c < 6; c++) wk += snew[c] * de[c];
        ea.wint += double(wd * R(0.5) * wk);
        tet4_forces<R>(Ji, snew, wd, put);
      } else {
        yielding = true;
      }
    } else {
      tet4_core<R, PHYS, true, STREAM>(p, at, get, dt, e, put, ea, &pre);
      if constexpr (PHYS == PHYS_EP) has_ep = pre.ep > R(0);
    }
  }
  if constexpr (PHYS == PHYS_EP) {
    const unsigned long long nb = __ballot(has_ep);
    if (has_word && (t & 63) == 0 && nb != yw) p.yielded[yi] = nb;
  }
  if constexpr (PHYS == PHYS_EP_MLP) {
    // rank of each yielding element in thread order
    const uint64_t m = __ballot(yielding);
    if (lane == 0) wcnt[w] = __popcll(m);
    __syncthreads();
    int total = 0, off = 0;
#pragma unroll
    for (int i = 0; i < NT / 64; i++) {
      const int c = wcnt[i];
      off += i < w ? c : 0;
      total += c;
    }
    const int rank = off + __popcll(m & ((1ull << lane) - 1ull));
    if constexpr (!WALK) {
      if (total > 0) {
        // nothing of the block has reached global memory yet: list it and
        // queue its yielding points' network inputs
        if (t == 0) {
          const unsigned long long old =
              atomicAdd(p.mlp_ctr, (1ull << 32) | (unsigned long long)total);
          p.mlp_list[old >> 32] = make_int2(b, (int)(unsigned)old);
          misc[0] = (unsigned)old;
        }
        __syncthreads();
        if (yielding) {
          float x[kMlpIn];
          mlp_inputs<R>(*p.mlp, de, pre.s, pre.ep, x);
          mlp_store_inputs(p.mlp_rows + (size_t)(misc[0] + rank) * kMlpRowHalves, x);
        }
        return;
      }
      // stored here, not last: held through the node pass, the stress
      // would not fit the elastic pass's 64 VGPRs
      if (has_e) store_state<STREAM, R>(at, snew, pre.ep, false);
    } else {
      int how = MLP_ELASTIC;
      if (yielding) {
        // the element again from the LDS node records (the same bits as
        // above; counted there), so nothing of it stays live across the
        // return map
        R Jy[9], dy[6], wy, sy[6];
        EAcc again;
        tet4_kin<R, PHYS_EP_MLP>(p, get, dt, Jy, dy, wy, again);
        R wky = ep_trial<R>(p, dy, pre.s, sy);
        R ep = pre.ep;
        const R q = yield_overshoot<R>(p, sy, ep);
        float y[kMlpOut];
        mlp_load_outputs(p.mlp_rows + (size_t)(qbase + rank) * kMlpRowHalves, y);
        const R dg = mlp_apply<R>(p, y, q, ep, sy, how);
#pragma unroll
        for (int c = 0; c < 6; c++) wky += sy[c] * dy[c];
        ea.wint += double(wy * R(0.5) * wky);
        if (dg > R(0))
          ea.wpl += double(wy * R(0.81649658092772603273) * (R(p.sy0) + R(p.H) * ep) * dg);
        tet4_forces<R>(Jy, sy, wy, put);
#pragma unroll
        for (int c = 0; c < 6; c++) snew[c] = sy[c];
        pre.ep = ep;
        ep_changed = true;
      }
      mlp_count(misc, how == MLP_ACCEPTED, how == MLP_FALLBACK);
      __syncthreads();
      if (t == 0 && p.mlp_stats && (misc[0] | misc[1])) {
        p.mlp_stats[2L * b] += misc[0];
        p.mlp_stats[2L * b + 1] += misc[1];
      }
    }
  } else {
    __syncthreads();
  }

  if (has_n) {
    double f[3];
    node_force_sum<R>(lf, joff, t, deg, f);
    if (slot < 0) {
      double x[3], v[3];
      ln.get(t, x, v);
      node_update<AUX != 0>(p, g, f, x, v, ln.mass(t), dt, ea);
    } else {
      store_partial<R>(p, slot, f);
    }
  }
  wave_flush<AUX != 0>(p, p.epart_base + b * (NT / 64), ea, row);
  // the walk stores the element's state last: registers that a store
  // reads must not be reused before it completes, so a store issued
  // earlier would hold up the node pass (the exact-return body stores it
  // in point_stress: held to the end, the FP64 kernel ran 1-2% slower)
  if constexpr (PHYS == PHYS_EP_MLP && WALK) {
    if (has_e) store_state<STREAM, R>(at, snew, pre.ep, ep_changed);
  }
}

template <typename R, int PHYS, int AUX, int NT, int WPE, bool STREAM, bool CW>
__global__ void __launch_bounds__(NT) __attribute__((amdgpu_waves_per_eu(WPE)))
k_elem_block4(Params p) {
  __shared__ int wcnt[NT / 64];
  __shared__ unsigned misc[2];
  block4<R, PHYS, AUX, NT, false, STREAM, CW>(p, xcd_remap(blockIdx.x, gridDim.x), 0u, wcnt, misc);
}

// The surrogate step's third launch: one workgroup per block of the grid,
// workgroup i finishing the i-th deferred block listed this step, if there
// is one, so the hardware spreads a plastic zone over the CUs as it would
// the blocks of an element pass (the list order depends on atomic order,
// the results of a block do not).  A loop over several listed blocks per
// workgroup holds the kernel arguments in SGPRs across iterations and
// spills 40-50 VGPRs.
template <bool AUX, int NT, int WPE, bool STREAM, bool CW>
__global__ void __launch_bounds__(NT) __attribute__((amdgpu_waves_per_eu(WPE)))
k_elem_block4_walk(Params p) {
  __shared__ int wcnt[NT / 64];
  __shared__ unsigned misc[2];
  if (blockIdx.x >= (unsigned)(*p.mlp_ctr >> 32)) return;
  const int2 ent = p.mlp_list[blockIdx.x];
  block4<float, PHYS_EP_MLP, AUX, NT, true, STREAM, CW>(
      p, __builtin_amdgcn_readfirstlane(ent.x), (unsigned)ent.y, wcnt, misc);
}

// The network on queue rows [0, n): n from the step's counter (ctr) or
// given.  Each workgroup with a tile to do copies the weights into LDS;
// its waves take tiles w, w + waves, ..., each reading the next tile's
// inputs before it runs the network on the current one, so the row loads
// (rows the previous launch wrote, from another XCD's L2 at best) overlap
// the MFMA chain.
template <int NT>
__global__ void __launch_bounds__(NT) k_mlp_queue(const MlpParams *P, uint16_t *rows,
                                                  const unsigned long long *ctr, int n_given) {
  __shared__ __attribute__((aligned(16))) MlpWeights W;
  constexpr int WPB = NT / 64;
  const unsigned n = ctr ? (unsigned)(*ctr & 0xffffffffull) : (unsigned)n_given;
  const int ntiles = (int)((n + 15u) >> 4);
  if ((int)blockIdx.x * WPB >= ntiles) return;
  mlp_lds_load(P->weights, &W);
  const int stride = (int)gridDim.x * WPB;
  int tile = (int)blockIdx.x * WPB + (int)(threadIdx.x >> 6);
  bf16x8 xb = mlp_tile_inputs(rows + (size_t)(tile < ntiles ? tile : 0) * 16 * kMlpRowHalves);
  __syncthreads();
  for (; tile < ntiles; tile += stride) {
    const int next = tile + stride < ntiles ? tile + stride : tile;
    const bf16x8 xn = mlp_tile_inputs(rows + (size_t)next * 16 * kMlpRowHalves);
    mlp_tile(W, xb, rows + (size_t)tile * 16 * kMlpRowHalves);
    xb = xn;
  }
}

// force records [s, s1) added to f in order, loaded four at a time
template <typename PR, typename I>
__device__ __forceinline__ void sum_records(const PR *rec, I s, I s1, double f[3]) {
  auto add = [&](const PR &q) {
    f[0] += double(q.x);
    f[1] += double(q.y);
    f[2] += double(q.z);
  };
  for (; s + 4 <= s1; s += 4) {
    const PR q0 = rec[s], q1 = rec[s + 1], q2 = rec[s + 2], q3 = rec[s + 3];
    add(q0);
    add(q1);
    add(q2);
    add(q3);
  }
  if (s + 2 <= s1) {
    const PR q0 = rec[s], q1 = rec[s + 1];
    add(q0);
    add(q1);
    s += 2;
  }
  if (s < s1) add(rec[s]);
}

template <int AUX, typename R>
__global__ void __launch_bounds__(256) k_node_bnd(Params p) {
  using PR = typename std::conditional<std::is_same<R, float>::value, Vec3f, Vec3>::type;
  const PR *part = reinterpret_cast<const PR *>(p.partial);
  const int i = xcd_remap(blockIdx.x, gridDim.x) * 256 + threadIdx.x;
  const RowPre row = row_prefetch(p, p.epart_base + blockIdx.x * 4);
  const double dt = p.ctl->dt;
  const bool leave = left_out<AUX>(p);
  EAcc ea;
  if (i < p.n_boundary) {
    const int g = p.n_interior + i;
    const Vec3 xr = p.pos[g], vv = p.vv[g];
    const double m = p.m[g];
    // partials in slot order
    double f[3] = {0.0, 0.0, 0.0};
    sum_records(part, p.slot_ptr[i], p.slot_ptr[i + 1], f);
    const double x[3] = {xr.x, xr.y, xr.z}, v[3] = {vv.x, vv.y, vv.z};
    if (!leave) node_update<AUX != 0>(p, g, f, x, v, m, dt, ea);
  }
  if (leave) return;
  wave_flush<AUX != 0>(p, p.epart_base + blockIdx.x * 4, ea, row);
  // the last launch of the step: the surrogate's queue and block list start
  // empty in the next one
  if (blockIdx.x == 0 && threadIdx.x == 0) {
    p.ctl->step += 1;
    if (p.mlp_ctr) *p.mlp_ctr = 0ull;
  }
}

// ---------------------------------------------------------------------------
// Resident steps: many steps of a mesh whose element blocks all fit the chip
// at once, in one launch.
//
// A small mesh spends its step on two launches and on the loads behind them
// (a 16-block mesh: 5.6 + 4.5 us for 0.7 MB that sits in the caches).  Here
// every block keeps its elements' stress state in registers and its node
// records in LDS from the first step to the last, and only the partial forces
// of shared nodes travel between blocks.
//
// Exchange.  A block posts its partial force on a shared node to every other
// block that holds the node, one message each, into the receiver's inbox
// (build_mail); each receiver adds the node's partials in slot order
// (k_node_bnd's order) and updates its own copy of the node, so all copies
// stay the same bits and no second launch, flag or grid barrier is needed.
// The messages between two blocks lie together, in the same order on both
// sides, and message m is posted and read by thread m of its block, so posts
// and inbox reads coalesce into whole lines: they are written and read past
// the XCDs' L2s (agent scope, sc1), where every transaction counts.  An empty
// message holds a NaN with a payload no arithmetic makes (MailRec::empty) in
// every word: the data is its own flag, word by word.  The reader empties a
// message as soon as it has it.  Steps alternate between two inboxes: the
// writer fills one again two steps later, after it has received the reader's
// message for the same node of the step between, which the reader posted
// after the emptying store completed (every thread waits for its stores
// before the barrier ahead of the posts).  A launch starts at the inbox after
// the last one's (base).
//
// All blocks have to run at once: a cooperative launch sized by
// resident_capacity.  Should some not get to run all the same (another
// process's kernels hold the chip), nothing hangs and nothing is lost: past
// spin_limit polls a thread decides that the launch gives up
// (Ctl::decision), and every block leaves without storing anything.  The
// blocks store their state only after the last of them to finish has decided
// that the launch counts, so a launch takes all its steps or none.  Until the
// host has seen to it (settled_ctl, which takes the missing steps with the
// per-step kernels), the later launches and the steps with outputs queued
// behind one that gave up are left out: what they would record belongs to
// later steps.
//
// Same arithmetic in the same order as the per-step kernels: same state
// bits.  The cumulative energies are summed over the steps per lane and over
// the lanes once at the end, shared nodes' by the block of their first slot.
//
// Per step (MI355X; before: the two launches): 6,000 tet4 8.9 -> 5.0 us
// (FP64), 8.7 -> 4.6 (FP32); 196,608 tet4 12.2 -> 7.9, 10.6 -> 6.5; 48,000 tet10
// 17.2 -> 10.3, 13.8 -> 8.7; 13,464 tet10 on the 5-point rule 12.4 -> 9.2, 12.3 ->
// 8.5.  What is left is the element pass and node sums
// (3.9 us for 16 blocks, 4.8 for 512) and one trip of the mail.
// ---------------------------------------------------------------------------
typedef unsigned mail4 __attribute__((ext_vector_type(4)));
typedef unsigned mail2 __attribute__((ext_vector_type(2)));
constexpr int kSc1 = 16;  // cache policy bit of the buffer builtins

// Message records, n of them: 16 bytes (x, y, z, unused) for FP32 partials;
// for FP64 ones (x, y) in 16 bytes and, past the n of those, z in 8.  Each word
// is an aligned 4- or 8-byte part of one store.
template <typename R> struct MailRec;
template <> struct MailRec<float> {
  static constexpr int bytes = 16;
  static constexpr unsigned empty = 0xffc0deadu, nan = 0x7fc00000u;
  __device__ static unsigned bits(float v) {
    const unsigned w = __float_as_uint(v);
    return w == empty ? nan : w;
  }
  __device__ static void put(__amdgpu_buffer_rsrc_t m, int, int i, const float f[3]) {
    const mail4 w = {bits(f[0]), bits(f[1]), bits(f[2]), 0u};
    __builtin_amdgcn_raw_buffer_store_b128(w, m, 16 * i, 0, kSc1);
  }
  __device__ static void clear(__amdgpu_buffer_rsrc_t m, int, int i) {
    const mail4 w = {empty, empty, empty, empty};
    __builtin_amdgcn_raw_buffer_store_b128(w, m, 16 * i, 0, kSc1);
  }
  __device__ static bool get(__amdgpu_buffer_rsrc_t m, int, int i, float f[3]) {
    const mail4 w = __builtin_amdgcn_raw_buffer_load_b128(m, 16 * i, 0, kSc1);
    f[0] = __uint_as_float(w.x);
    f[1] = __uint_as_float(w.y);
    f[2] = __uint_as_float(w.z);
    return w.x != empty && w.y != empty && w.z != empty;
  }
};
template <> struct MailRec<double> {
  static constexpr int bytes = 24;
  static constexpr unsigned long long empty = 0xfff8dead5107e000ull, nan = 0x7ff8000000000000ull;
  __device__ static unsigned long long bits(double v) {
    const unsigned long long w = (unsigned long long)__double_as_longlong(v);
    return w == empty ? nan : w;
  }
  __device__ static void store(__amdgpu_buffer_rsrc_t m, int n, int i, unsigned long long x,
                               unsigned long long y, unsigned long long z) {
    const mail4 a = {(unsigned)x, (unsigned)(x >> 32), (unsigned)y, (unsigned)(y >> 32)};
    const mail2 b = {(unsigned)z, (unsigned)(z >> 32)};
    __builtin_amdgcn_raw_buffer_store_b128(a, m, 16 * i, 0, kSc1);
    __builtin_amdgcn_raw_buffer_store_b64(b, m, 8 * i, 16 * n, kSc1);
  }
  __device__ static void put(__amdgpu_buffer_rsrc_t m, int n, int i, const double f[3]) {
    store(m, n, i, bits(f[0]), bits(f[1]), bits(f[2]));
  }
  __device__ static void clear(__amdgpu_buffer_rsrc_t m, int n, int i) {
    store(m, n, i, empty, empty, empty);
  }
  __device__ static bool get(__amdgpu_buffer_rsrc_t m, int n, int i, double f[3]) {
    const mail4 a = __builtin_amdgcn_raw_buffer_load_b128(m, 16 * i, 0, kSc1);
    const mail2 b = __builtin_amdgcn_raw_buffer_load_b64(m, 8 * i, 16 * n, kSc1);
    const unsigned long long x = a.x | (unsigned long long)a.y << 32,
                             y = a.z | (unsigned long long)a.w << 32,
                             z = b.x | (unsigned long long)b.y << 32;
    f[0] = __longlong_as_double((long long)x);
    f[1] = __longlong_as_double((long long)y);
    f[2] = __longlong_as_double((long long)z);
    return x != empty && y != empty && z != empty;
  }
};

__device__ __forceinline__ __amdgpu_buffer_rsrc_t mail_rsrc(void *mail, int bytes) {
  return __builtin_amdgcn_make_buffer_rsrc(mail, 0, bytes, 0x00027000);
}

template <typename R>
__global__ void __launch_bounds__(256) k_mail_clear(void *mail, int records) {
  const int i = blockIdx.x * 256 + threadIdx.x;
  if (i < records) MailRec<R>::clear(mail_rsrc(mail, records * MailRec<R>::bytes), records, i);
}

// LDS past the element kernel's: the messages received, then per message its
// destination, its local node and the nodes' message lists
__host__ __device__ constexpr int lds_mail_bytes(int rsz, int most) {
  return lds_round16(3L * rsz * most) + lds_round16(8L * most);
}

__device__ __forceinline__ uint32_t decision(const Params &p) {
  return __hip_atomic_load(&p.ctl->decision, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
}
// launch L's decision, taken once: 0 it counts, 1 it gives up
__device__ __forceinline__ void decide(const Params &p, unsigned L, unsigned how) {
  atomicCAS(&p.ctl->decision, 2u * (L - 1u), 2u * L + how);
}

// Thread t has node t of the block, and the element and point that it has in the
// per-step kernels: tet4, element t (k_elem_block4); tet10 on a 4-point rule,
// PointLane's (k_elem_block10); on the five-point rule, point lane % 5 of the
// wave's element lane / 5, twelve of them (k_elem_block5).
template <int NPE, int RULE, typename R, int PHYS, int NT, int WPE>
__global__ void __launch_bounds__(NT) __attribute__((amdgpu_waves_per_eu(WPE)))
k_resident(Params p, Resident rs) {
  using Rec = MailRec<R>;
  extern __shared__ double smem[];
  __shared__ int gave_up;
  // after a launch that gave up, whose mail lies about, none runs
  if (threadIdx.x == 0) gave_up = decision(p) & 1u;
  __syncthreads();
  if (gave_up) return;
  const int b = xcd_remap(blockIdx.x, gridDim.x);
  const int t = threadIdx.x;
  // the thread's element and point, as the per-step kernels take them
  constexpr bool FIVE = NPE == 10 && Quad<RULE>::n == 5;
  constexpr bool MM = NPE == 10 && !FIVE && sizeof(R) == 8;
  const PointLane<MM> pt(t);
  const int lane = t & 63;
  const int q = NPE == 4 ? 0 : FIVE ? lane % 5 : pt.q;
  const int el = NPE == 4 ? t : FIVE ? 12 * (t >> 6) + lane / 5 : pt.el;
  auto place = [&]() { return NPE == 4 ? t : FIVE ? 5 * el + q : pt.place(p); };
  const int32_t *mt = p.meta + 8 * b;
  const int es = mt[0], nel = mt[1];
  const LNodes ln{smem, p.ml};
  R *lf = (R *)((char *)smem + lds_node_bytes(p.ml));
  uint16_t *joff = (uint16_t *)((char *)lf + lds_force_bytes(sizeof(R), NPE, p.max_el));
  double *basis = (double *)((char *)joff + lds_off_bytes(p.kmax));
  R *lm = (R *)((char *)basis + lds_basis_bytes(NPE, sizeof(R), Quad<RULE>::n));
  int32_t *ldest = (int32_t *)((char *)lm + lds_round16(3L * sizeof(R) * rs.most));
  uint16_t *lsrc = (uint16_t *)(ldest + rs.most), *lidx = lsrc + rs.most;
  const double dt = p.ctl->dt;
  const int wv = __builtin_amdgcn_readfirstlane(t >> 6);
  const bool has_word = PHYS == PHYS_EP && wv < p.ywords;
  const long yi = (long)b * p.ywords + wv;

  // Node t: its record, and in two registers its contribution count, its
  // place among the blocks holding it, its messages (kNotShared: none, and
  // this block alone moves it) and their start in the list.
  constexpr unsigned kNotShared = 0xffffu;
  const long o = (long)b * p.ml + t;
  const int g = t < p.ml ? p.nid_pad[o] : -1;
  const bool has_n = g >= 0;
  unsigned deg_lo = 0u, own_cnt = kNotShared << 16;
  bool held = false, contact = false;
  if (has_n) {
    held = node_held(p, g);
    contact = node_contact(p, g, held);
    const int slot = p.slot_pad[o];
    deg_lo = p.deg_pad[o];
    if (slot >= 0) {
      const int s0 = p.slot_ptr[g - p.n_interior], s1 = p.slot_ptr[g - p.n_interior + 1];
      deg_lo |= (unsigned)rs.lo[o] << 16;
      own_cnt = (unsigned)(slot - s0) | (unsigned)(s1 - s0 - 1) << 16;
    }
    ln.stage(t, p.pos[g], p.m[g], p.vv[g]);
  }
  const int m0 = rs.first[b], nm = rs.first[b + 1] - m0;
  for (int m = t; m < nm; m += NT) {
    ldest[m] = rs.dest[m0 + m];
    lsrc[m] = rs.src[m0 + m];
    lidx[m] = rs.idx[m0 + m];
  }
  const __amdgpu_buffer_rsrc_t mail = mail_rsrc(rs.mail, (int)(2 * rs.messages * Rec::bytes));
  for (int k = t; k <= p.kmax; k += NT) joff[k] = p.off_pad[(long)b * (p.kmax + 1) + k];
  if constexpr (MM)
    for (int k = t; k < Tet10Basis<RULE>::n; k += NT) basis[k] = tet10_basis<RULE>.v[k];
  // element el: corner words and the point's state
  const bool has_e = el < nel && (!FIVE || lane < 60);
  uint32_t cw[NPE / 2];
  PreState<R> pre{};
  {
    const int ec = es + (has_e ? el : nel - 1);
    const uint32_t *cp = reinterpret_cast<const uint32_t *>(p.corner + (long)NPE * ec);
#pragma unroll
    for (int k = 0; k < NPE / 2; k++) cw[k] = cp[k];
  }
  if (has_e) {
    if constexpr (PHYS == PHYS_EP) {
      const unsigned long long yw = has_word ? p.yielded[yi] : FIVE ? ~0ull : 0ull;
      load_state<false, R>(state_block<R>(p, b, place()), (yw >> (t & 63)) & 1ull, pre);
    }
  }
  __syncthreads();

  EAcc ea;
  bool changed = false;
  auto half = [&](int k) { return (int)((cw[k >> 1] >> (16 * (k & 1))) & 0xffffu); };
  auto get = [&](int k, double xk[3], double vk[3]) { ln.get(half(k) & 511, xk, vk); };
  auto slot_of = [&](int h) { return (int)joff[h >> 9] + (h & 511); };
  int box = rs.base;  // the step's inbox, 0 or 1
  int qs = q, ts = t;
  ParamsAt args = params_at();
  for (int left = rs.steps; left > 0; left--, box ^= 1) {
    // What follows from the lane's point, node and corners (basis values, LDS
    // addresses) is cheap to form and must not be held over the step: hoisted
    // out of the loop it costs 30 to 90 spilled registers.
    asm volatile("" : "+v"(qs), "+v"(ts), "+v"(deg_lo), "+v"(own_cnt));
#pragma unroll
    for (int k = 0; k < NPE / 2; k++) asm volatile("" : "+v"(cw[k]));
    Params pl = params_again(args, p);
    pl.samples = nullptr;  // the recorder's steps are not resident
    if constexpr (NPE == 4) {
      if (has_e) {
        auto put = [&](int k, const R fk[3]) {
          R *dst = lf + 3 * slot_of(half(k));
#pragma unroll
          for (int c = 0; c < 3; c++) dst[c] = fk[c];
        };
        tet4_core<R, PHYS, true, false, true>(pl, StatePlane<R>{}, get, dt, es + el, put, ea, &pre);
      }
    } else if constexpr (FIVE) {
      auto slot = [&](int k) { return slot_of(half(k)); };
      if (has_e)
        tet10_five<RULE, R, PHYS, true>(pl, StatePlane<R>{}, get, slot, lf, dt, es + el, qs, pre, ea);
    } else {
      tet10_block<RULE, R, PHYS, false, true, MM>(pl, StatePlane<R>{}, ln, lf, joff, basis, cw, dt,
                                              es + el, ts, qs, has_e, el - (t & 15) < nel, pre, ea);
    }
    if constexpr (PHYS == PHYS_EP)
      if (has_e) changed = changed || pre.changed;
    // the emptying stores of the last step have completed
    asm volatile("s_waitcnt vmcnt(0)" ::: "memory");
    __syncthreads();
    double f[3];
    if (has_n) {
      node_force_sum<R>(lf, joff, ts, (int)(deg_lo & 0xffffu), f);
      // the partial for the posts, in the node's own first slot (off[0] = 0)
      if ((own_cnt >> 16) != kNotShared) {
#pragma unroll
        for (int c = 0; c < 3; c++) lf[3 * ts + c] = R(f[c]);
      }
    }
    __syncthreads();
    const int inbox = box * rs.messages;
    for (int m = ts; m < nm; m += NT) {
      const R *fs = lf + 3 * lsrc[m];
      const R fr[3] = {fs[0], fs[1], fs[2]};
      Rec::put(mail, 2 * rs.messages, inbox + ldest[m], fr);
    }
    for (int m = ts; m < nm; m += NT) {
      R w[3];
      unsigned spins = 0;
      // (decision by p: pl's pointer would be loaded again ahead of every wait,
      // 3% of a step of 3,072 tet4 in FP32)
      while (!Rec::get(mail, 2 * rs.messages, inbox + m0 + m, w)) {
        if (++spins >= rs.spin_limit || ((spins & 255u) == 0u && (decision(p) & 1u))) {
          gave_up = 1;
          break;
        }
        asm volatile("" ::: "memory");
      }
      Rec::clear(mail, 2 * rs.messages, inbox + m0 + m);
#pragma unroll
      for (int c = 0; c < 3; c++) lm[3 * m + c] = w[c];
    }
    __syncthreads();
    if (gave_up) break;
    if (has_n) {
      const int own = (int)(own_cnt & 0xffffu), cnt = (int)(own_cnt >> 16);
      if (cnt != (int)kNotShared) {
        const int lo = (int)(deg_lo >> 16);
        double s[3] = {0.0, 0.0, 0.0};
        auto add = [&](int k) {
          const R *msg = lm + 3 * lidx[lo + k];
#pragma unroll
          for (int c = 0; c < 3; c++) s[c] += double(msg[c]);
        };
        for (int k = 0; k < own; k++) add(k);
#pragma unroll
        for (int c = 0; c < 3; c++) s[c] += f[c];
        for (int k = own; k < cnt; k++) add(k);
#pragma unroll
        for (int c = 0; c < 3; c++) f[c] = s[c];
      }
      double x[3], v[3];
      ln.get(ts, x, v);
      const double m = ln.mass(ts);
      NodeStep s;
      EAcc en;
      node_advance(pl, held, contact, f, x, v, m, 1.0 / m, dt, s, en);
      if (own == 0) ea.wgrav += en.wgrav;
      ln.stage(ts, Vec3{s.x[0], s.x[1], s.x[2]}, m, Vec3{s.v[0], s.v[1], s.v[2]});
    }
    __syncthreads();
  }

  // all blocks or none
  if (gridDim.x > 1) {
    if (t == 0 && gave_up) {
      decide(p, rs.launch, 1u);
    } else if (t == 0) {
      const uint64_t all = (uint64_t)rs.launch * gridDim.x;
      if (atomicAdd((unsigned long long *)&p.ctl->finished, 1ull) + 1ull == all)
        decide(p, rs.launch, 0u);
      uint32_t d = decision(p);
      for (unsigned spins = 0; d == 2u * (rs.launch - 1u); d = decision(p))
        if (++spins == rs.spin_limit) decide(p, rs.launch, 1u);
      gave_up = d & 1u;
    }
    __syncthreads();
    if (gave_up) return;
  } else if (t == 0) {
    decide(p, rs.launch, 0u);
  }
  if (has_n && (own_cnt & 0xffffu) == 0u) {
    const int n = p.nid_pad[o];
    double x[3], v[3];
    ln.get(t, x, v);
    p.pos[n] = Vec3{x[0], x[1], x[2]};
    p.vv[n] = Vec3{v[0], v[1], v[2]};
  }
  if constexpr (PHYS == PHYS_EP) {
    if (has_e) store_state<false, R>(state_block<R>(p, b, place()), pre.s, pre.ep, changed);
    const unsigned long long nb = __ballot(has_e && pre.ep > R(0));
    if (has_word && (t & 63) == 0) p.yielded[yi] = nb;
  }
  const int row_base = p.epart_base + b * (NT / 64);
  wave_flush<false>(p, row_base, ea, row_prefetch(p, row_base));
  if (blockIdx.x == 0 && t == 0) {
    p.ctl->step += rs.steps;
    p.ctl->resident += rs.steps;
  }
}

// The nodes of no element, the last ones: no block holds one, and only gravity
// and the wall act on them, so each takes a resident launch's steps by itself,
// once the launch counts.
__global__ void __launch_bounds__(256) k_resident_loose(Params p, Resident rs) {
  const int g = p.nn - rs.loose + (int)(blockIdx.x * 256 + threadIdx.x);
  if (g >= p.nn || p.ctl->decision != 2u * rs.launch) return;
  const bool held = node_held(p, g), contact = node_contact(p, g, held);
  const double f[3] = {0.0, 0.0, 0.0}, m = p.m[g], dt = p.ctl->dt;
  const Vec3 xr = p.pos[g], vr = p.vv[g];
  double x[3] = {xr.x, xr.y, xr.z}, v[3] = {vr.x, vr.y, vr.z};
  for (int k = 0; k < rs.steps; k++) {
    NodeStep s;
    EAcc ea;  // without mass there is no energy
    node_advance(p, held, contact, f, x, v, m, 1.0 / m, dt, s, ea);
#pragma unroll
    for (int c = 0; c < 3; c++) {
      x[c] = s.x[c];
      v[c] = s.v[c];
    }
  }
  p.pos[g] = Vec3{x[0], x[1], x[2]};
  p.vv[g] = Vec3{v[0], v[1], v[2]};
}

// ---------------------------------------------------------------------------
// colour / atomic element pass: one thread per element, nodes from HBM
//
// Colour: the forces go to per-node slots, summed by k_node_all in ascending
// colour, the order in which one launch per colour would add them, so the
// sums have the same bits.  One launch per colour (30 of them on a box mesh)
// costs a launch and a chain of dependent loads each, for a few thousand
// elements; the slots cost 24 (FP32: 12) bytes written and read per corner.
// Per step: 6,000 tet4 148 -> 10.0 us, 48,000 tet10 684 -> 35 us, 1.57M
// tet4 484 -> 204 us (there bound by the scattered 24-byte records).
// ---------------------------------------------------------------------------
// Atomic: on n elements, those of list if it is given.  One launch per colour
// is the colour scatter of a mesh whose slots found no room: each node takes at
// most one sum per launch, so the order and the bits are the same.
template <int NPE, int RULE, typename R, int PHYS, bool ATOMIC, int NT>
__global__ void __launch_bounds__(NT) k_elem_direct(Params p, const int32_t *list, int n) {
  using FR = typename std::conditional<std::is_same<R, float>::value, Vec3f, Vec3>::type;
  const int t = blockIdx.x * NT + threadIdx.x;
  const RowPre row = row_prefetch(p, p.epart_base + blockIdx.x * (NT / 64));
  const double dt = p.ctl->dt;
  EAcc ea;
  if (t < n) {
    const int e = ATOMIC && list ? list[t] : t;
    int nd[NPE];
#pragma unroll
    for (int k = 0; k < NPE; k++) nd[k] = p.conn[(long)k * p.ne + e];
    auto get = [&](int k, double xk[3], double vk[3]) {
      const Vec3 a = p.pos[nd[k]], b = p.vv[nd[k]];
      xk[0] = a.x;
      xk[1] = a.y;
      xk[2] = a.z;
      vk[0] = b.x;
      vk[1] = b.y;
      vk[2] = b.z;
    };
    auto put = [&](int k, const R fk[3]) {
      if constexpr (ATOMIC) {
#pragma unroll
        for (int c = 0; c < 3; c++) unsafeAtomicAdd(&p.f[c][nd[k]], double(fk[c]));
      } else {
        static_cast<FR *>(p.cforce)[p.fslot[(long)k * p.ne + e]] = FR{fk[0], fk[1], fk[2]};
      }
    };
    elem_core<NPE, RULE, R, PHYS>(p, get, dt, e, put, ea);
  }
  wave_flush<true>(p, p.epart_base + blockIdx.x * (NT / 64), ea, row);
}

// FR: the record of a corner-force slot (colour scatter), or void for the
// sums of the atomic scatter, which are cleared for the next step
template <bool AUX, typename FR>
__global__ void __launch_bounds__(256) k_node_all(Params p) {
  const int g = blockIdx.x * 256 + threadIdx.x;
  const RowPre row = row_prefetch(p, p.epart_base + blockIdx.x * 4);
  const double dt = p.ctl->dt;
  EAcc ea;
  if (g < p.nn) {
    const Vec3 xr = p.pos[g], vv = p.vv[g];
    const double m = p.m[g];
    double f[3] = {0.0, 0.0, 0.0};
    if constexpr (std::is_void<FR>::value) {
#pragma unroll
      for (int c = 0; c < 3; c++) {
        f[c] = p.f[c][g];
        p.f[c][g] = 0.0;
      }
    } else {
      sum_records(static_cast<const FR *>(p.cforce), p.node_slot[g], p.node_slot[g + 1], f);
    }
    const double x[3] = {xr.x, xr.y, xr.z}, v[3] = {vv.x, vv.y, vv.z};
    node_update<AUX>(p, g, f, x, v, m, dt, ea);
  }
  wave_flush<AUX>(p, p.epart_base + blockIdx.x * 4, ea, row);
  if (blockIdx.x == 0 && threadIdx.x == 0) p.ctl->step += 1;
}

// initial update with du = 0 (f_int = 0) and the half-kick
// (dynamics.h:454-463): a0 = wall(X0) + g; v += dt/2 a0
__global__ void __launch_bounds__(256) k_node_init(Params p) {
  const int g = blockIdx.x * 256 + threadIdx.x;
  const RowPre row = row_prefetch(p, blockIdx.x * 4);
  const double dt = p.ctl->dt;
  EAcc ea;
  if (g < p.nn) {
    const Vec3 xr = p.pos[g], vv = p.vv[g];
    const double m = p.m[g];
    const bool held = p.fixed_mask && p.fixed_mask[g];
    const double x[3] = {xr.x, xr.y, xr.z};
    const double v[3] = {held ? 0.0 : vv.x, held ? 0.0 : vv.y, held ? 0.0 : vv.z};
    double a[3] = {0.0, 0.0, 0.0}, ke = 0.0, vn[3];
    if (p.wall_on && !held && (!p.contact_mask || p.contact_mask[g])) {
#pragma unroll
      for (int c = 0; c < 3; c++)
        if (c == p.wall_dim) {
          double d = (x[c] - p.wall_loc) * p.wall_normal;
          if (d < 0.0) {
            a[c] += -1 * (1 / m) * d * p.wall_nk;
            ea.pen += 0.5 * p.wall_k * d * d;
            ea.fc += -p.wall_k * d;
          }
        }
    }
#pragma unroll
    for (int c = 0; c < 3; c++) {
      a[c] = held ? 0.0 : a[c] + p.grav[c];
      ke += v[c] * v[c];
      vn[c] = v[c] + 0.5 * dt * a[c];
    }
    p.vv[g] = Vec3{vn[0], vn[1], vn[2]};
    p.acc[g] = Node4{a[0], a[1], a[2], 0.0};
    p.du[g] = Node4{0.0, 0.0, 0.0, 0.0};
    p.xprev[g] = Node4{xr.x, xr.y, xr.z, m};
    ea.ke = 0.5 * m * ke;
  }
  wave_flush<true>(p, blockIdx.x * 4, ea, row);
}

// Energy rows are summed in two fixed-order stages: kEredBlocks workgroups
// each reduce a contiguous chunk of rows into p.ered, then one wave sums
// those and writes the energy row of this step.
constexpr int kEredBlocks = 64;

__global__ void __launch_bounds__(256) k_energy_reduce1(Params p) {
  __shared__ double red[256 * EP_N];
  const int chunk = (p.n_epart + kEredBlocks - 1) / kEredBlocks;
  const int r0 = blockIdx.x * chunk, r1 = min(p.n_epart, r0 + chunk);
  double v[EP_N] = {0, 0, 1e300, 0, 0, 0, 0, 0};
  for (int r = r0 + threadIdx.x; r < r1; r += 256) {
    const double *src = p.epart + (long)r * EP_N;
    // a stable-dt entry of 0 is a row no kernel has written since the rows
    // were cleared (cpi_init's own reduction, rows only the half-kick
    // writes); it takes no part in the minimum.  A degenerate element
    // (limit 0) is caught by the inverted-element count instead.
#pragma unroll
    for (int k = 0; k < EP_N; k++)
      v[k] = (k == EP_MINDT) ? fmin(v[k], src[k] > 0.0 ? src[k] : 1e300) : v[k] + src[k];
  }
#pragma unroll
  for (int k = 0; k < EP_N; k++) red[threadIdx.x * EP_N + k] = v[k];
  __syncthreads();
  for (int h = 128; h > 0; h >>= 1) {
    if ((int)threadIdx.x < h)
#pragma unroll
      for (int k = 0; k < EP_N; k++) {
        double o = red[(threadIdx.x + h) * EP_N + k];
        double &d = red[threadIdx.x * EP_N + k];
        d = (k == EP_MINDT) ? fmin(d, o) : d + o;
      }
    __syncthreads();
  }
  if (threadIdx.x < EP_N) p.ered[blockIdx.x * EP_N + threadIdx.x] = red[threadIdx.x];
}

__global__ void __launch_bounds__(64) k_energy_reduce2(Params p) {
  if (threadIdx.x == 0) {
    const bool leave = left_out<STEP_OUT_ASK>(p);  // (0 without resident steps)
    double s[EP_N] = {0, 0, 1e300, 0, 0, 0, 0, 0};
    for (int b = 0; b < kEredBlocks; b++)
      for (int k = 0; k < EP_N; k++) {
        const double o = p.ered[b * EP_N + k];
        s[k] = (k == EP_MINDT) ? fmin(s[k], o) : s[k] + o;
      }
    if (leave) return;
    Ctl *c = p.ctl;
    double row[8];
    row[0] = s[EP_KE];
    row[1] = s[EP_WINT];
    row[2] = s[EP_WPL];
    row[3] = s[EP_PEN];
    row[4] = s[EP_WGRAV];
    row[5] = s[EP_FC];
    if (c->step == 0) c->e0 = row[0] + row[3];
    row[6] = row[0] + row[1] + row[3] - row[4] - c->e0;
    row[7] = s[EP_MINDT];
    bool finite = true;
    for (int k = 0; k < 7; k++) {
      c->row[k] = row[k];
      finite = finite && isfinite(row[k]);
    }
    c->row[7] = row[7];
    if (!finite) c->flags |= 1u;
    if (s[EP_BAD] > 0.0) c->flags |= 2u;
    // the elastoplastic kernels reduce the element CFL limit of the
    // configuration each step started from (the others leave 1e300): a
    // fixed dt above it, or above the wall spring's limit, is unstable
    if (row[7] < 1e300 && !(c->dt <= fmin(row[7], c->dt_contact))) c->flags |= 4u;
    if (p.hist && p.hist_cap > 0) {
      double *h = p.hist + (c->nrows % p.hist_cap) * 8;
      for (int k = 0; k < 8; k++) h[k] = row[k];
      c->nrows += 1;
    }
  }
}

// ---------------------------------------------------------------------------
// lumped mass, into m
// ---------------------------------------------------------------------------
template <int NPE, int RULE, int NT>
__global__ void __launch_bounds__(NT) k_mass_block(Params p, int kind, double rho) {
  extern __shared__ double smem[];
  const int b = blockIdx.x;
  const int32_t *mt = p.meta + 8 * b;
  const int es = mt[0], nel = mt[1];
  const int ml = p.ml;
  const int32_t *nid = p.nid_pad + (long)b * ml;
  double *lx = smem;               // x, y, z: ml each
  double *lm = smem + 3 * ml;      // corner masses, jagged-diagonal slots
  uint16_t *joff = (uint16_t *)(lm + (long)p.max_el * NPE);
  for (int j = threadIdx.x; j < ml; j += NT) {
    const int g = nid[j];
    if (g >= 0) {
      const Vec3 q = p.pos[g];
      lx[j] = q.x;
      lx[ml + j] = q.y;
      lx[2 * ml + j] = q.z;
    }
  }
  for (int k = threadIdx.x; k <= p.kmax; k += NT) joff[k] = p.off_pad[(long)b * (p.kmax + 1) + k];
  __syncthreads();
  for (int t = threadIdx.x; t < nel; t += NT) {
    const int e = es + t;
    double xs[NPE][3], me[NPE];
#pragma unroll
    for (int k = 0; k < NPE; k++) {
      const int l = p.conn_local[(long)e * NPE + k];
#pragma unroll
      for (int c = 0; c < 3; c++) xs[k][c] = lx[c * ml + l];
    }
    elem_mass<NPE, RULE>(xs, kind, rho, me);
#pragma unroll
    for (int k = 0; k < NPE; k++) lm[p.csr_pos[(long)e * NPE + k]] = me[k];
  }
  __syncthreads();
  for (int j = threadIdx.x; j < ml; j += NT) {
    const int g = nid[j];
    if (g < 0) continue;
    double sum = 0.0;
    const int deg = p.deg_pad[(long)b * ml + j];
    for (int k = 0; k < deg; k++) sum += lm[joff[k] + j];
    const int slot = p.slot_pad[(long)b * ml + j];
    if (slot < 0)
      p.m[g] = sum;
    else
      p.partial[slot].x = sum;
  }
}

__global__ void __launch_bounds__(256) k_mass_bnd(Params p) {
  const int i = blockIdx.x * 256 + threadIdx.x;
  if (i >= p.n_boundary) return;
  double s = 0.0;
  for (int q = p.slot_ptr[i]; q < p.slot_ptr[i + 1]; q++) s += p.partial[q].x;
  p.m[p.n_interior + i] = s;
}

// colour scatter: corner masses into the x of the corner-force slots (FP64
// words, whatever the slots' record), summed in colour order by k_mass_slots
// (atomic: on n elements, those of list if it is given, as k_elem_direct)
template <int NPE, int RULE, bool ATOMIC>
__global__ void __launch_bounds__(256) k_mass_direct(Params p, int kind, double rho,
                                                      const int32_t *list, int n) {
  const int t = blockIdx.x * 256 + threadIdx.x;
  if (t >= n) return;
  const int e = ATOMIC && list ? list[t] : t;
  int nd[NPE];
  double xs[NPE][3], me[NPE];
#pragma unroll
  for (int k = 0; k < NPE; k++) {
    nd[k] = p.conn[(long)k * p.ne + e];
    const Vec3 q = p.pos[nd[k]];
    xs[k][0] = q.x;
    xs[k][1] = q.y;
    xs[k][2] = q.z;
  }
  elem_mass<NPE, RULE>(xs, kind, rho, me);
#pragma unroll
  for (int k = 0; k < NPE; k++) {
    if (ATOMIC)
      unsafeAtomicAdd(&p.m[nd[k]], me[k]);
    else
      static_cast<double *>(p.cforce)[p.fslot[(long)k * p.ne + e]] = me[k];
  }
}

__global__ void __launch_bounds__(256) k_mass_slots(Params p) {
  const int g = blockIdx.x * 256 + threadIdx.x;
  if (g >= p.nn) return;
  double s = 0.0;
  for (uint32_t q = p.node_slot[g]; q < p.node_slot[g + 1]; q++)
    s += static_cast<const double *>(p.cforce)[q];
  p.m[g] = s;
}

// ---------------------------------------------------------------------------
// stable dt of the current configuration, one minimum per workgroup
// ---------------------------------------------------------------------------
template <int NPE>
__global__ void __launch_bounds__(256) k_elem_dt(Params p, double *out) {
  __shared__ double red[4];
  const int e = blockIdx.x * 256 + threadIdx.x;
  double d = 1e300;
  if (e < p.ne) {
    double xs[4][3];
#pragma unroll
    for (int k = 0; k < 4; k++) {
      const Vec3 q = p.pos[p.conn[(long)k * p.ne + e]];
      xs[k][0] = q.x;
      xs[k][1] = q.y;
      xs[k][2] = q.z;
    }
    // linear corner order: tet4 (0,1,2,3); tet10 corners (2,0,1,3)
    const int o = NPE == 4 ? 0 : 2, i1 = NPE == 4 ? 1 : 0, i2 = NPE == 4 ? 2 : 1;
    double e1[3], e2[3], e3[3];
#pragma unroll
    for (int c = 0; c < 3; c++) {
      e1[c] = xs[i1][c] - xs[o][c];
      e2[c] = xs[i2][c] - xs[o][c];
      e3[c] = xs[3][c] - xs[o][c];
    }
    double v6 = e1[0] * (e2[1] * e3[2] - e2[2] * e3[1]) - e1[1] * (e2[0] * e3[2] - e2[2] * e3[0]) +
                e1[2] * (e2[0] * e3[1] - e2[1] * e3[0]);
    d = corner_dt<double>(e1, e2, e3, v6, p.wave_speed,
                          NPE == 4 ? kTet4LengthFactor : kTet10LengthFactor);
  }
  d = wave_min(d);
  if ((threadIdx.x & 63) == 0) red[threadIdx.x >> 6] = d;
  __syncthreads();
  if (threadIdx.x == 0) out[blockIdx.x] = fmin(fmin(red[0], red[1]), fmin(red[2], red[3]));
}

// ---------------------------------------------------------------------------
// nodal strain/stress at xi = 0 from the total displacement x_n + du - X0
// with B(x_n) (dynamics_kernels.h:117-130, analysis.h:479-503)
// ---------------------------------------------------------------------------
// One thread per node, user order: a node takes the value of the
// highest-numbered element that holds it (last, a device element id, -1 for
// a node of none), so only that element is evaluated and only 96 bytes per
// node leave the device.  Evaluating every element and picking on the host
// moved 96 bytes per element, twice through host memory: an exported frame
// of 196,608 tet4 (100 FP32 steps, nodal state, strain and stress) took 11.8
// ms, now 1.9 ms.  Bound by the copy to the caller's pages.
template <int NPE>
__global__ void __launch_bounds__(256) k_stress_node(Params p, const int32_t *last, int count,
                                                     double *strain, double *stress) {
  const int node = blockIdx.x * 256 + threadIdx.x;
  if (node >= count) return;
  const int e = last[node];
  if (e < 0) return;
  double xs[NPE][3], u[NPE][3];
#pragma unroll
  for (int k = 0; k < NPE; k++) {
    const int n = p.conn[(long)k * p.ne + e];
    const Node4 xp = p.xprev[n], d = p.du[n], x0 = p.X0[n];
    xs[k][0] = xp.x;
    xs[k][1] = xp.y;
    xs[k][2] = xp.z;
    u[k][0] = d.x + xp.x - x0.x;
    u[k][1] = d.y + xp.y - x0.y;
    u[k][2] = d.z + xp.z - x0.z;
  }
  double G[NPE * 3];
  if constexpr (NPE == 4) {
    const double g4[12] = {-1, -1, -1, 1, 0, 0, 0, 1, 0, 0, 0, 1};
#pragma unroll
    for (int i = 0; i < 12; i++) G[i] = g4[i];
  } else {
    tet10_grad(0.0, 0.0, 0.0, G);
  }
  double J[9] = {0, 0, 0, 0, 0, 0, 0, 0, 0};
#pragma unroll
  for (int i = 0; i < NPE; i++)
#pragma unroll
    for (int a = 0; a < 3; a++)
#pragma unroll
      for (int c = 0; c < 3; c++) J[a * 3 + c] += G[3 * i + c] * xs[i][a];
  double Ji[9];
  inv3<double>(J, Ji);
  double de[6] = {0, 0, 0, 0, 0, 0};
#pragma unroll
  for (int i = 0; i < NPE; i++) {
    double dn[3];
#pragma unroll
    for (int c = 0; c < 3; c++)
      dn[c] = Ji[c] * G[3 * i] + Ji[3 + c] * G[3 * i + 1] + Ji[6 + c] * G[3 * i + 2];
    de[0] += dn[0] * u[i][0];
    de[1] += dn[1] * u[i][1];
    de[2] += dn[2] * u[i][2];
    de[3] += dn[1] * u[i][0] + dn[0] * u[i][1];
    de[4] += dn[2] * u[i][1] + dn[1] * u[i][2];
    de[5] += dn[2] * u[i][0] + dn[0] * u[i][2];
  }
  if (strain) {
    double *o = strain + 6L * node;
#pragma unroll
    for (int c = 0; c < 6; c++) o[c] = de[c];
  }
  if (!stress) return;
  double *o = stress + 6L * node;
  o[0] = p.c11 * de[0] + p.c12 * (de[1] + de[2]);
  o[1] = p.c11 * de[1] + p.c12 * (de[0] + de[2]);
  o[2] = p.c11 * de[2] + p.c12 * (de[0] + de[1]);
  o[3] = p.c44 * de[3];
  o[4] = p.c44 * de[4];
  o[5] = p.c44 * de[5];
}

// ---------------------------------------------------------------------------
// known-answer strain energy and volume on the reference positions
// (dynamics.h:303-412, analysis.h:384-477): W_e = 1/2 sum_q w detJ de.D.de,
// V_e = sum_q w detJ
// ---------------------------------------------------------------------------
template <int NPE, int RULE>
__global__ void __launch_bounds__(256) k_debug_strain(Params p, double alpha, int dcase,
                                                       double nu, double *out) {
  __shared__ double red[8];
  const int e = blockIdx.x * 256 + threadIdx.x;
  double W = 0.0, V = 0.0;
  if (e < p.ne) {
    double xs[NPE][3], u[NPE][3];
#pragma unroll
    for (int k = 0; k < NPE; k++) {
      const Node4 q = p.X0[p.conn[(long)k * p.ne + e]];
      xs[k][0] = q.x;
      xs[k][1] = q.y;
      xs[k][2] = q.z;
      const double x = q.x;
      const double s = dcase == 0 ? alpha * x : alpha * 0.5 * x * x;
      u[k][0] = s;
      u[k][1] = -s * nu;
      u[k][2] = -s * nu;
    }
#pragma unroll
    for (int q = 0; q < Quad<RULE>::n; q++) {
      double G[NPE * 3];
      if constexpr (NPE == 4) {
        const double g4[12] = {-1, -1, -1, 1, 0, 0, 0, 1, 0, 0, 0, 1};
#pragma unroll
        for (int i = 0; i < 12; i++) G[i] = g4[i];
      } else {
        tet10_grad(Quad<RULE>::pt(q, 0), Quad<RULE>::pt(q, 1), Quad<RULE>::pt(q, 2), G);
      }
      double J[9] = {0, 0, 0, 0, 0, 0, 0, 0, 0};
#pragma unroll
      for (int i = 0; i < NPE; i++)
#pragma unroll
        for (int a = 0; a < 3; a++)
#pragma unroll
          for (int c = 0; c < 3; c++) J[a * 3 + c] += G[3 * i + c] * xs[i][a];
      double Ji[9];
      double detJ = inv3<double>(J, Ji);
      double de[6] = {0, 0, 0, 0, 0, 0};
#pragma unroll
      for (int i = 0; i < NPE; i++) {
        double dn[3];
#pragma unroll
        for (int c = 0; c < 3; c++)
          dn[c] = Ji[c] * G[3 * i] + Ji[3 + c] * G[3 * i + 1] + Ji[6 + c] * G[3 * i + 2];
        de[0] += dn[0] * u[i][0];
        de[1] += dn[1] * u[i][1];
        de[2] += dn[2] * u[i][2];
        de[3] += dn[1] * u[i][0] + dn[0] * u[i][1];
        de[4] += dn[2] * u[i][1] + dn[1] * u[i][2];
        de[5] += dn[2] * u[i][0] + dn[0] * u[i][2];
      }
      double s0 = p.c11 * de[0] + p.c12 * (de[1] + de[2]);
      double s1 = p.c11 * de[1] + p.c12 * (de[0] + de[2]);
      double s2 = p.c11 * de[2] + p.c12 * (de[0] + de[1]);
      double w = Quad<RULE>::w(q) * detJ;
      W += 0.5 * w *
           (s0 * de[0] + s1 * de[1] + s2 * de[2] +
            p.c44 * (de[3] * de[3] + de[4] * de[4] + de[5] * de[5]));
      V += w;
    }
  }
  W = wave_sum(W);
  V = wave_sum(V);
  if ((threadIdx.x & 63) == 0) {
    red[2 * (threadIdx.x >> 6)] = W;
    red[2 * (threadIdx.x >> 6) + 1] = V;
  }
  __syncthreads();
  if (threadIdx.x == 0) {
    out[2 * blockIdx.x] = red[0] + red[2] + red[4] + red[6];
    out[2 * blockIdx.x + 1] = red[1] + red[3] + red[5] + red[7];
  }
}

// ---------------------------------------------------------------------------
// host layouts: user-order [N][3] arrays to and from the device's node
// records, user-order element state from the device's structure of arrays.
// One thread per double of the host array, so the host side is contiguous
// across a wave and the records are gathered 24 bytes at a time; permuting on
// the host cost several passes over fresh host pages per array.
// ---------------------------------------------------------------------------
__global__ void __launch_bounds__(256) k_import_nodes(const double *src, const int32_t *ninv,
                                                      int n, Vec3 *d3, Node4 *d4) {
  const long i = (long)blockIdx.x * 256 + threadIdx.x;
  if (i >= 3L * n) return;
  const int k = (int)(i / 3), c = (int)(i - 3L * k);
  const long g = ninv[k];
  const double v = src[i];
  if (d3) reinterpret_cast<double *>(d3)[3 * g + c] = v;
  if (d4) {
    reinterpret_cast<double *>(d4)[4 * g + c] = v;
    if (c == 0) d4[g].w = 0.0;
  }
}

// ctl: a copy of the control block, so one transfer brings it along
__global__ void __launch_bounds__(256) k_export_nodes(Params p, const int32_t *ninv, int n,
                                                      NodeExport o) {
  const long i = (long)blockIdx.x * 256 + threadIdx.x;
  constexpr int words = sizeof(Ctl) / 8;
  if (blockIdx.x == 0 && threadIdx.x < words && o.ctl)
    reinterpret_cast<uint64_t *>(o.ctl)[threadIdx.x] =
        reinterpret_cast<const uint64_t *>(p.ctl)[threadIdx.x];
  if (i >= 3L * n) return;
  const int k = (int)(i / 3), c = (int)(i - 3L * k);
  const long g = ninv[k];
  if (o.x) o.x[i] = reinterpret_cast<const double *>(p.pos)[3 * g + c];
  double v = 0.0, a = 0.0;
  if (o.v || o.vi) v = reinterpret_cast<const double *>(p.vv)[3 * g + c];
  if (o.a || o.vi) a = reinterpret_cast<const double *>(p.acc)[4 * g + c];
  if (o.v) o.v[i] = v;
  if (o.a) o.a[i] = a;
  if (o.vi) {
    // v_n = v_{n+1/2} - dt/2 a_n, product and difference rounded apart
    const double h = o.half_dt * a;
    o.vi[i] = v - h;
  }
  if (o.m && c == 0) o.m[k] = p.m[g];
  if (o.m3) o.m3[i] = p.m[g];
}

// place in ep (and in a component of sig) of point q of an element.  spos, of
// the element: in the planes (state_ld 0) the device element; in rows per
// block its place in elements, and its points lie next to each other, or
// (p.matrix) as PointLane<true> places them
__device__ __forceinline__ long state_place(const Params &p, uint32_t spos, int q) {
  if (!p.state_ld) return spos + (long)q * p.ne;
  if (!p.matrix) return (long)spos * p.nq + q;
  const uint32_t w = p.state_ld < 64 ? p.state_ld >> 2 : 16;
  return (long)(spos / w) * 4 * w + q * w + spos % w;
}

template <typename R>
__global__ void __launch_bounds__(256) k_export_elems(Params p, const uint32_t *spos, int n,
                                                      double *sig, double *ep) {
  const long i = (long)blockIdx.x * 256 + threadIdx.x, ne = p.ne, ld = p.state_ld;
  const int w = 6 * p.nq;
  if (sig && i < (long)n * w) {
    const long e = i / w;
    const int q = (int)(i - e * w) / 6, c = (int)(i - e * w) - 6 * q;
    const long at = state_place(p, spos[e], q);
    const R *sr = static_cast<const R *>(p.sig);
    sig[i] = double(ld ? sr[(at / ld) * 6 * ld + c * ld + at % ld]
                       : sr[(6L * q + c) * ne + spos[e]]);
  }
  if (ep && i < (long)n * p.nq) {
    const long e = i / p.nq;
    const int q = (int)(i - e * p.nq);
    ep[i] = double(static_cast<const R *>(p.epbar)[state_place(p, spos[e], q)]);
  }
}

// x = X0, v = v0, du, a and the assembled forces (atomic scatter) zeroed
__global__ void __launch_bounds__(256) k_reset_nodes(Params p, const Vec3 *v0) {
  const int g = blockIdx.x * 256 + threadIdx.x;
  if (g >= p.nn) return;
  const Node4 x = p.X0[g];
  p.pos[g] = Vec3{x.x, x.y, x.z};
  p.vv[g] = v0[g];
  p.xprev[g] = Node4{x.x, x.y, x.z, 0.0};
  p.acc[g] = Node4{0.0, 0.0, 0.0, 0.0};
  p.du[g] = Node4{0.0, 0.0, 0.0, 0.0};
  if (p.f[0] == nullptr) return;
#pragma unroll
  for (int c = 0; c < 3; c++) p.f[c][g] = 0.0;
}

// the smallest positive mass, one value per workgroup (1e300: none)
__global__ void __launch_bounds__(256) k_mass_min(const double *m, int nn, double *out) {
  __shared__ double red[4];
  double v = 1e300;
  for (int i = blockIdx.x * 256 + threadIdx.x; i < nn; i += (int)gridDim.x * 256)
    if (m[i] > 0.0) v = fmin(v, m[i]);
  v = wave_min(v);
  if ((threadIdx.x & 63) == 0) red[threadIdx.x >> 6] = v;
  __syncthreads();
  if (threadIdx.x == 0) out[blockIdx.x] = fmin(fmin(red[0], red[1]), fmin(red[2], red[3]));
}

// ---------------------------------------------------------------------------
// streaming copy (bandwidth probe and counter calibration)
// ---------------------------------------------------------------------------
__global__ void __launch_bounds__(256) k_stream_copy(const Node4 *__restrict__ src,
                                                     Node4 *__restrict__ dst, long n) {
  const long stride = (long)gridDim.x * 256;
  for (long i = (long)blockIdx.x * 256 + threadIdx.x; i < n; i += stride) dst[i] = src[i];
}

// ---------------------------------------------------------------------------
// launchers
// ---------------------------------------------------------------------------

// Events the next element or node kernel launch records at its own start
// and end (hipExtLaunchKernel), for cpi_profile_kernels: the kernel's
// execution time without the event packets' own latency.  Null: a plain
// launch.  Per host thread.
static thread_local hipEvent_t t_ev_start = nullptr, t_ev_stop = nullptr;

void set_launch_events(hipEvent_t start, hipEvent_t stop) {
  t_ev_start = start;
  t_ev_stop = stop;
}

template <typename K, typename... A>
static inline void timed_launch(K kern, dim3 grid, dim3 block, size_t smem, hipStream_t s,
                                A... args) {
  if (t_ev_start || t_ev_stop)
    hipExtLaunchKernelGGL(kern, grid, block, (std::uint32_t)smem, s, t_ev_start, t_ev_stop, 0,
                          args...);
  else
    hipLaunchKernelGGL(kern, grid, block, smem, s, args...);
}

#define CPI_LAUNCH(kern, grid, block, smem, stream, ...)                      \
  do {                                                                        \
    timed_launch((kern), dim3(grid), dim3(block), (smem), (stream), __VA_ARGS__); \
    return hipGetLastError();                                                 \
  } while (0)

// threads per workgroup of the block kernels: tet4 one per element (384),
// tet10 one per point (512 for 128 elements; on the five-point rule, twelve
// elements per wave, 704)
template <int NPE, int RULE> constexpr int block_threads() {
  return NPE == 4 ? 384 : (Quad<RULE>::n == 4 ? 512 : 704);
}
// default elements per workgroup
constexpr int block_elements(int npe) { return npe == 4 ? 384 : 128; }
// minimum waves per SIMD of the per-point tet10 kernel
template <typename R> constexpr int tet10_waves() { return 4; }

// Threads of the 5-point tet10 kernel (cus: the device's CUs).  Up to one block per CU a step takes
// as long as one block does, and 704 threads do its 128 elements in one round
// (13k elements, FP64 compat: 9.5 us, 384 threads 12.2).  With more blocks 384
// threads, two rounds, leave room for more workgroups per CU and one's loads
// overlap another's arithmetic (663k elements: FP64 compat 141 us against 153,
// FP32 114 against 139, FP32 EP 154 against 170), but FP64 EP takes 148 VGPRs,
// three waves per SIMD, where a second 6-wave workgroup often finds no room:
// 259 us against 230.
constexpr int kNarrow5 = 384;
template <typename R, int PHYS> constexpr bool may_narrow5() {
  return sizeof(R) == 4 || PHYS == PHYS_COMPAT;
}
static bool narrow5(int nblocks, int cus, bool f64_state) { return nblocks > cus && !f64_state; }
// its waves per SIMD: FP64 with a state takes 148 VGPRs
template <typename R, int PHYS> constexpr int tet10_waves5() {
  return sizeof(R) == 8 && PHYS != PHYS_COMPAT ? 3 : 4;
}

// minimum waves per SIMD the tet4 element kernels are compiled for: FP64
// fits 96 VGPRs (three 6-wave workgroups per CU), FP32 64 (five per CU);
// the surrogate step's elastic pass has the plain FP32 kernel's structure
// and budget.  Its walk (network outputs, acceptance checks, the FP64
// fallback) spills 19 VGPRs at 64 and none at 80: six waves per SIMD, four
// workgroups per CU.
template <typename R, int PHYS> constexpr int tet4_waves() {
  return std::is_same<R, double>::value ? 5 : 8;
}
constexpr int kMlpWalkWaves = 6;

// workgroups of k_mlp_queue in the step (four waves each, every wave
// looping over tiles): eight per CU, eight waves per SIMD at 32 VGPRs and
// 15 KB of LDS each
constexpr int kMlpQueueGrid = 2048;
constexpr int kMlpQueueThreads = 256;

// LDS of the workgroup element kernels: node records, corner forces, the
// slot offsets, the basis of the FP64 per-point tet10 kernels
size_t elem_block_smem(int npe, int rule, int prec, int ml, int max_el, int kmax) {
  const int rsz = prec == 1 ? 4 : 8;
  return (size_t)lds_node_bytes(ml) + lds_force_bytes(rsz, npe, max_el) + lds_off_bytes(kmax) +
         lds_basis_bytes(npe, rsz, rule == RULE_REF5 ? 5 : 4);
}

int elem_block_threads(int npe, int rule, int prec, int phys, int nblocks, int cus) {
  if (npe == 4) return block_threads<4, RULE_CENTROID>();
  if (rule == RULE_REF5)
    return narrow5(nblocks, cus, prec != 1 && phys != PHYS_COMPAT) ? kNarrow5
                                                                   : block_threads<10, RULE_REF5>();
  return block_threads<10, RULE_EXACT4>();
}

int elem_block_default_elements(int npe) { return block_elements(npe); }

// dynamic LDS above 64 KiB needs an explicit opt-in per kernel
template <typename K>
static hipError_t lds_opt_in(K kernel, size_t smem) {
  if (smem <= 65536) return hipSuccess;
  return hipFuncSetAttribute(reinterpret_cast<const void *>(kernel),
                             hipFuncAttributeMaxDynamicSharedMemorySize, (int)smem);
}

// the tet4 kernels' LDS opt-in, cached or streamed state, corner words or
// the two u16 arrays
template <typename R, int PHYS, bool STREAM, bool CW>
static hipError_t tet4_opt_in(size_t smem) {
  constexpr int NT = block_threads<4, RULE_CENTROID>();
  constexpr int W = tet4_waves<R, PHYS>();
  hipError_t e = lds_opt_in(k_elem_block4<R, PHYS, STEP_OUT, NT, W, STREAM, CW>, smem);
  if (e == hipSuccess) e = lds_opt_in(k_elem_block4<R, PHYS, STEP_PLAIN, NT, W, STREAM, CW>, smem);
  if constexpr (CW && PHYS != PHYS_EP_MLP)
    if (e == hipSuccess)
      e = lds_opt_in(k_elem_block4<R, PHYS, STEP_OUT_ASK, NT, W, STREAM, CW>, smem);
  if constexpr (PHYS == PHYS_EP_MLP) {
    if (e == hipSuccess)
      e = lds_opt_in(k_elem_block4_walk<true, NT, kMlpWalkWaves, STREAM, CW>, smem);
    if (e == hipSuccess)
      e = lds_opt_in(k_elem_block4_walk<false, NT, kMlpWalkWaves, STREAM, CW>, smem);
  }
  return e;
}

// the LDS opt-in (prepare_elem_block) is done once at set-up, outside any
// stream capture
// the tet4 launches, with the stress state cached or streamed (STREAM),
// the corners as 16-bit words or two u16 arrays (CW)
template <typename R, int PHYS, bool STREAM, bool CW>
static hipError_t elem_block4_t(const Params &p, bool aux, int nblocks, size_t smem,
                                hipStream_t s, int part) {
  constexpr int NT = block_threads<4, RULE_CENTROID>();
  constexpr int W = tet4_waves<R, PHYS>();
  if constexpr (PHYS == PHYS_EP_MLP) {
    // the elastic pass, the network on the queue, the walk over the
    // deferred blocks (part 1, 2, 3 alone for per-launch timing)
    if (part == 0 || part == 1) {
      if (aux)
        timed_launch((k_elem_block4<R, PHYS, STEP_OUT, NT, W, STREAM, CW>), dim3(nblocks), dim3(NT),
                     smem, s, p);
      else
        timed_launch((k_elem_block4<R, PHYS, STEP_PLAIN, NT, W, STREAM, CW>), dim3(nblocks), dim3(NT),
                     smem, s, p);
    }
    if (part == 0 || part == 2) {
      const int tiles = (p.ne + 15) / 16;
      const int grid = std::max(1, std::min(kMlpQueueGrid, (tiles + 3) / 4));
      timed_launch((k_mlp_queue<kMlpQueueThreads>), dim3(grid), dim3(kMlpQueueThreads), 0, s,
                   p.mlp, p.mlp_rows, (const unsigned long long *)p.mlp_ctr, 0);
    }
    if (part == 0 || part == 3) {
      const int grid = nblocks;
      if (aux)
        timed_launch((k_elem_block4_walk<true, NT, kMlpWalkWaves, STREAM, CW>), dim3(grid), dim3(NT),
                     smem, s, p);
      else
        timed_launch((k_elem_block4_walk<false, NT, kMlpWalkWaves, STREAM, CW>), dim3(grid), dim3(NT),
                     smem, s, p);
    }
    return hipGetLastError();
  } else {
    if constexpr (CW)
      if (aux && p.resident)
        CPI_LAUNCH((k_elem_block4<R, PHYS, STEP_OUT_ASK, NT, W, STREAM, CW>), nblocks, NT, smem, s, p);
    if (aux) CPI_LAUNCH((k_elem_block4<R, PHYS, STEP_OUT, NT, W, STREAM, CW>), nblocks, NT, smem, s, p);
    CPI_LAUNCH((k_elem_block4<R, PHYS, STEP_PLAIN, NT, W, STREAM, CW>), nblocks, NT, smem, s, p);
  }
}

// the per-point tet10 kernel's LDS opt-in and launch, cached or streamed
// state, quads or the matrix units (p.matrix)
template <int RULE, typename R, int PHYS, bool STREAM, bool MM>
static hipError_t tet10_opt_in(size_t smem) {
  constexpr int NT = block_threads<10, RULE>();
  constexpr int W = tet10_waves<R>();
  hipError_t e = lds_opt_in(k_elem_block10<RULE, R, PHYS, STEP_OUT, NT, W, STREAM, MM>, smem);
  if (e == hipSuccess)
    e = lds_opt_in(k_elem_block10<RULE, R, PHYS, STEP_PLAIN, NT, W, STREAM, MM>, smem);
  if constexpr (MM || sizeof(R) == 4)
    if (e == hipSuccess)
      e = lds_opt_in(k_elem_block10<RULE, R, PHYS, STEP_OUT_ASK, NT, W, STREAM, MM>, smem);
  return e;
}

template <int RULE, typename R, int PHYS, bool STREAM, bool MM>
static hipError_t tet10_t(const Params &p, bool aux, int nblocks, size_t smem, hipStream_t s) {
  constexpr int NT = block_threads<10, RULE>();
  constexpr int W = tet10_waves<R>();
  if constexpr (MM || sizeof(R) == 4)
    if (aux && p.resident)
      CPI_LAUNCH((k_elem_block10<RULE, R, PHYS, STEP_OUT_ASK, NT, W, STREAM, MM>), nblocks, NT, smem, s,
                 p);
  if (aux)
    CPI_LAUNCH((k_elem_block10<RULE, R, PHYS, STEP_OUT, NT, W, STREAM, MM>), nblocks, NT, smem, s, p);
  CPI_LAUNCH((k_elem_block10<RULE, R, PHYS, STEP_PLAIN, NT, W, STREAM, MM>), nblocks, NT, smem, s, p);
}

template <int NPE, int RULE, typename R, int PHYS>
static hipError_t elem_block_t(const Params &p, bool aux, int nblocks, size_t smem, hipStream_t s,
                               int part) {
  constexpr int NT = block_threads<NPE, RULE>();
  if constexpr (NPE == 4) {
    // a plan whose blocks exceed the corner words has none uploaded, and
    // its state cached
    if (!p.corner) return elem_block4_t<R, PHYS, false, false>(p, aux, nblocks, smem, s, part);
    if constexpr (PHYS != PHYS_COMPAT)
      if (p.stream_state) return elem_block4_t<R, PHYS, true, true>(p, aux, nblocks, smem, s, part);
    return elem_block4_t<R, PHYS, false, true>(p, aux, nblocks, smem, s, part);
  } else if constexpr (Quad<RULE>::n == 4) {
    if constexpr (sizeof(R) == 8) {
      if (p.matrix) {
        if constexpr (PHYS != PHYS_COMPAT)
          if (p.stream_state) return tet10_t<RULE, R, PHYS, true, true>(p, aux, nblocks, smem, s);
        return tet10_t<RULE, R, PHYS, false, true>(p, aux, nblocks, smem, s);
      }
    }
    if constexpr (PHYS != PHYS_COMPAT)
      if (p.stream_state) return tet10_t<RULE, R, PHYS, true, false>(p, aux, nblocks, smem, s);
    return tet10_t<RULE, R, PHYS, false, false>(p, aux, nblocks, smem, s);
  } else {
    constexpr int W = tet10_waves5<R, PHYS>();
    if constexpr (may_narrow5<R, PHYS>()) {
      constexpr int N2 = kNarrow5;
      if (p.narrow5) {
        if (aux) CPI_LAUNCH((k_elem_block5<RULE, R, PHYS, STEP_OUT, N2, W>), nblocks, N2, smem, s, p);
        CPI_LAUNCH((k_elem_block5<RULE, R, PHYS, STEP_PLAIN, N2, W>), nblocks, N2, smem, s, p);
      }
    }
    if (aux && p.resident)
      CPI_LAUNCH((k_elem_block5<RULE, R, PHYS, STEP_OUT_ASK, NT, W>), nblocks, NT, smem, s, p);
    if (aux) CPI_LAUNCH((k_elem_block5<RULE, R, PHYS, STEP_OUT, NT, W>), nblocks, NT, smem, s, p);
    CPI_LAUNCH((k_elem_block5<RULE, R, PHYS, STEP_PLAIN, NT, W>), nblocks, NT, smem, s, p);
  }
}

template <int NPE, int RULE, typename R, int PHYS>
static hipError_t elem_direct_t(const Params &p, bool atomic, const int32_t *list, int n,
                                hipStream_t s) {
  constexpr int NT = NPE == 4 ? 256 : 128;
  const int grid = (n + NT - 1) / NT;
  if (atomic) CPI_LAUNCH((k_elem_direct<NPE, RULE, R, PHYS, true, NT>), grid, NT, 0, s, p, list, n);
  CPI_LAUNCH((k_elem_direct<NPE, RULE, R, PHYS, false, NT>), grid, NT, 0, s, p, list, n);
}

int elem_direct_threads(int npe) { return npe == 4 ? 256 : 128; }

// (npe, rule, precision, physics) -> instantiation
template <template <int, int, typename, int> class F, typename... A>
static hipError_t dispatch(int npe, int rule, int prec, int phys, A &&...a) {
#define CPI_PHYS(NPE, RULE, R)                                         \
  switch (phys) {                                                      \
    case PHYS_COMPAT: return F<NPE, RULE, R, PHYS_COMPAT>::run(a...); \
    case PHYS_EP: return F<NPE, RULE, R, PHYS_EP>::run(a...);         \
    case PHYS_EP_MLP: return F<NPE, RULE, R, PHYS_EP_MLP>::run(a...); \
  }                                                                    \
  return hipErrorInvalidValue;
#define CPI_PREC(NPE, RULE)    \
  if (prec == 1) {             \
    CPI_PHYS(NPE, RULE, float) \
  } else {                     \
    CPI_PHYS(NPE, RULE, double) \
  }
  if (npe == 4) {
    CPI_PREC(4, RULE_CENTROID)
  }
  switch (rule) {
    case RULE_REF5: CPI_PREC(10, RULE_REF5)
    case RULE_REF4: CPI_PREC(10, RULE_REF4)
    case RULE_EXACT4: CPI_PREC(10, RULE_EXACT4)
  }
#undef CPI_PREC
#undef CPI_PHYS
  return hipErrorInvalidValue;
}

template <int NPE, typename R, int PHYS>
constexpr bool valid_combo() {
  return PHYS != PHYS_EP_MLP || (NPE == 4 && std::is_same<R, float>::value);
}

template <int NPE, int RULE, typename R, int PHYS> struct ElemBlockF {
  static hipError_t run(const Params &p, bool aux, int nb, size_t smem, hipStream_t s, int part) {
    if constexpr (!valid_combo<NPE, R, PHYS>())
      return hipErrorInvalidValue;
    else
      return elem_block_t<NPE, RULE, R, PHYS>(p, aux, nb, smem, s, part);
  }
};
template <int NPE, int RULE, typename R, int PHYS> struct ElemBlockPrepF {
  static hipError_t run(size_t smem) {
    if constexpr (!valid_combo<NPE, R, PHYS>()) {
      return hipErrorInvalidValue;
    } else {
      constexpr int NT = block_threads<NPE, RULE>();
      if constexpr (NPE == 4) {
        hipError_t e = tet4_opt_in<R, PHYS, false, true>(smem);
        if (e == hipSuccess) e = tet4_opt_in<R, PHYS, false, false>(smem);
        if constexpr (PHYS != PHYS_COMPAT)
          if (e == hipSuccess) e = tet4_opt_in<R, PHYS, true, true>(smem);
        return e;
      } else if constexpr (Quad<RULE>::n == 4) {
        hipError_t e = tet10_opt_in<RULE, R, PHYS, false, false>(smem);
        if constexpr (PHYS != PHYS_COMPAT)
          if (e == hipSuccess) e = tet10_opt_in<RULE, R, PHYS, true, false>(smem);
        if constexpr (sizeof(R) == 8) {
          if (e == hipSuccess) e = tet10_opt_in<RULE, R, PHYS, false, true>(smem);
          if constexpr (PHYS != PHYS_COMPAT)
            if (e == hipSuccess) e = tet10_opt_in<RULE, R, PHYS, true, true>(smem);
        }
        return e;
      } else {
        constexpr int W = tet10_waves5<R, PHYS>();
        hipError_t e = lds_opt_in(k_elem_block5<RULE, R, PHYS, STEP_OUT, NT, W>, smem);
        if (e == hipSuccess) e = lds_opt_in(k_elem_block5<RULE, R, PHYS, STEP_OUT_ASK, NT, W>, smem);
        if (e == hipSuccess) e = lds_opt_in(k_elem_block5<RULE, R, PHYS, STEP_PLAIN, NT, W>, smem);
        if constexpr (may_narrow5<R, PHYS>()) {
          if (e == hipSuccess)
            e = lds_opt_in(k_elem_block5<RULE, R, PHYS, STEP_OUT, kNarrow5, W>, smem);
          if (e == hipSuccess)
            e = lds_opt_in(k_elem_block5<RULE, R, PHYS, STEP_PLAIN, kNarrow5, W>, smem);
        }
        return e;
      }
    }
  }
};
template <int NPE, int RULE, typename R, int PHYS> struct ElemDirectF {
  static hipError_t run(const Params &p, bool atomic, const int32_t *list, int n, hipStream_t s) {
    if constexpr (PHYS == PHYS_EP_MLP)
      return hipErrorInvalidValue;
    else
      return elem_direct_t<NPE, RULE, R, PHYS>(p, atomic, list, n, s);
  }
};

hipError_t launch_elem_block(const Params &p, int rule, int prec, int phys, bool aux, int nblocks,
                             size_t smem, hipStream_t s, int part) {
  return dispatch<ElemBlockF>(p.npe, rule, prec, phys, p, aux, nblocks, smem, s, part);
}

hipError_t prepare_elem_block(int npe, int rule, int prec, int phys, size_t smem) {
  return dispatch<ElemBlockPrepF>(npe, rule, prec, phys, smem);
}

hipError_t launch_elem_direct(const Params &p, int rule, int prec, int phys, bool atomic,
                              const int32_t *list, int n, hipStream_t s) {
  return dispatch<ElemDirectF>(p.npe, rule, prec, phys, p, atomic, list, n, s);
}

// minimum waves per SIMD of the resident kernels: the five-point tet10 kernel's eleven waves a block
// leave a CU no second block, and get the registers
template <int NPE, int RULE> constexpr int resident_waves() {
  return NPE == 10 && Quad<RULE>::n == 5 ? 3 : 4;
}

hipError_t launch_resident_loose(const Params &p, const Resident &rs, hipStream_t s) {
  if (rs.loose == 0) return hipSuccess;
  CPI_LAUNCH(k_resident_loose, (rs.loose + 255) / 256, 256, 0, s, p, rs);
}

template <int NPE, int RULE, typename R, int PHYS> struct ResidentF {
  static constexpr bool has() {
    return PHYS != PHYS_EP_MLP;
  }
  // the kernel, its threads per workgroup
  static hipError_t run(const void **kernel, int *threads) {
    if constexpr (!has()) {
      return hipErrorInvalidValue;
    } else {
      *kernel = reinterpret_cast<const void *>(
          k_resident<NPE, RULE, R, PHYS, block_threads<NPE, RULE>(), resident_waves<NPE, RULE>()>);
      *threads = block_threads<NPE, RULE>();
      return hipSuccess;
    }
  }
};

int resident_capacity(int npe, int rule, int prec, int phys, size_t smem, int cus) {
  const void *k = nullptr;
  int nt = 0, per = 0;
  if (dispatch<ResidentF>(npe, rule, prec, phys, &k, &nt) != hipSuccess) return 0;
  if (smem > 65536 &&
      hipFuncSetAttribute(k, hipFuncAttributeMaxDynamicSharedMemorySize, (int)smem) != hipSuccess)
    return 0;
  if (hipOccupancyMaxActiveBlocksPerMultiprocessor(&per, k, nt, smem) != hipSuccess) return 0;
  // The query counts waves over the whole CU; a workgroup of six waves lands
  // as 2, 2, 1, 1 on the four SIMDs, and nothing makes the next one fill the
  // gaps.  Count ceil(waves / 4) on every SIMD, so that all really fit.
  hipFuncAttributes at{};
  if (hipFuncGetAttributes(&at, k) != hipSuccess || at.numRegs <= 0) return 0;
  const int simd = std::min(8, 512 / ((at.numRegs + 7) / 8 * 8)), wg = (nt / 64 + 3) / 4;
  return std::min(per, simd / wg) * cus;
}

hipError_t launch_resident(const Params &p, int rule, int prec, int phys, const Resident &rs,
                           int nblocks, size_t smem, hipStream_t s) {
  const void *k = nullptr;
  int nt = 0;
  hipError_t e = dispatch<ResidentF>(p.npe, rule, prec, phys, &k, &nt);
  if (e != hipSuccess) return e;
  Params pa = p;
  Resident ra = rs;
  void *args[2] = {&pa, &ra};
  // one block waits for nobody
  if (nblocks == 1) return hipLaunchKernel(k, dim3(1), dim3(nt), args, smem, s);
  return hipLaunchCooperativeKernel(k, dim3(nblocks), dim3(nt), args, (unsigned)smem, s);
}

hipError_t launch_mail_clear(const Resident &rs, int prec, hipStream_t s) {
  const int records = 2 * rs.messages;
  if (records == 0) return hipSuccess;
  if (prec == 1) CPI_LAUNCH(k_mail_clear<float>, (records + 255) / 256, 256, 0, s, rs.mail, records);
  CPI_LAUNCH(k_mail_clear<double>, (records + 255) / 256, 256, 0, s, rs.mail, records);
}

size_t resident_smem(size_t block_smem, int prec, int most) {
  return block_smem + lds_mail_bytes(prec == 1 ? 4 : 8, most);
}

size_t mail_bytes(int prec, size_t messages) {
  return 2 * messages * (prec == 1 ? MailRec<float>::bytes : MailRec<double>::bytes);
}

hipError_t launch_node_bnd(const Params &p, int prec, bool aux, hipStream_t s) {
  const int grid = std::max(1, (p.n_boundary + 255) / 256);
  if (aux && p.resident) {
    if (prec == 1) CPI_LAUNCH((k_node_bnd<STEP_OUT_ASK, float>), grid, 256, 0, s, p);
    CPI_LAUNCH((k_node_bnd<STEP_OUT_ASK, double>), grid, 256, 0, s, p);
  }
  if (prec == 1) {
    if (aux) CPI_LAUNCH((k_node_bnd<STEP_OUT, float>), grid, 256, 0, s, p);
    CPI_LAUNCH((k_node_bnd<STEP_PLAIN, float>), grid, 256, 0, s, p);
  }
  if (aux) CPI_LAUNCH((k_node_bnd<STEP_OUT, double>), grid, 256, 0, s, p);
  CPI_LAUNCH((k_node_bnd<STEP_PLAIN, double>), grid, 256, 0, s, p);
}

hipError_t launch_node_all(const Params &p, int prec, bool aux, hipStream_t s) {
  const int grid = (p.nn + 255) / 256;
  if (!p.cforce) {
    if (aux) CPI_LAUNCH((k_node_all<true, void>), grid, 256, 0, s, p);
    CPI_LAUNCH((k_node_all<false, void>), grid, 256, 0, s, p);
  }
  if (prec == 1) {
    if (aux) CPI_LAUNCH((k_node_all<true, Vec3f>), grid, 256, 0, s, p);
    CPI_LAUNCH((k_node_all<false, Vec3f>), grid, 256, 0, s, p);
  }
  if (aux) CPI_LAUNCH((k_node_all<true, Vec3>), grid, 256, 0, s, p);
  CPI_LAUNCH((k_node_all<false, Vec3>), grid, 256, 0, s, p);
}

hipError_t launch_node_init(const Params &p, hipStream_t s) {
  CPI_LAUNCH(k_node_init, (p.nn + 255) / 256, 256, 0, s, p);
}

hipError_t launch_energy_reduce(const Params &p, hipStream_t s) {
  hipLaunchKernelGGL(k_energy_reduce1, dim3(kEredBlocks), dim3(256), 0, s, p);
  hipError_t e = hipGetLastError();
  if (e != hipSuccess) return e;
  CPI_LAUNCH(k_energy_reduce2, 1, 64, 0, s, p);
}

int energy_reduce_blocks() { return kEredBlocks; }

template <int NPE, int RULE>
static hipError_t mass_rule_t(const Params &p, int scatter, int kind, double rho, int nblocks,
                              const int32_t *list, int n, hipStream_t s) {
  if (scatter == 0) {
    constexpr int NT = NPE == 4 ? 512 : 128;
    const size_t smem = 8 * (3 * (size_t)p.ml + (size_t)p.max_el * NPE) + lds_off_bytes(p.kmax);
    if (smem > 65536) return hipErrorInvalidValue;  // sized by the plan to stay below
    hipLaunchKernelGGL((k_mass_block<NPE, RULE, NT>), dim3(nblocks), dim3(NT), smem, s, p, kind,
                       rho);
    hipError_t e = hipGetLastError();
    if (e != hipSuccess || p.n_boundary == 0) return e;
    CPI_LAUNCH(k_mass_bnd, (p.n_boundary + 255) / 256, 256, 0, s, p);
  }
  const int grid = (n + 255) / 256;
  if (scatter == 2)
    CPI_LAUNCH((k_mass_direct<NPE, RULE, true>), grid, 256, 0, s, p, kind, rho, list, n);
  hipLaunchKernelGGL((k_mass_direct<NPE, RULE, false>), dim3(grid), dim3(256), 0, s, p, kind, rho,
                     list, n);
  hipError_t e = hipGetLastError();
  if (e != hipSuccess) return e;
  CPI_LAUNCH(k_mass_slots, (p.nn + 255) / 256, 256, 0, s, p);
}

hipError_t launch_mass(const Params &p, int rule, int scatter, int kind, double rho, int nblocks,
                       const int32_t *list, int n, hipStream_t s) {
  if (p.npe == 4) {
    switch (rule) {
      case RULE_REF4: return mass_rule_t<4, RULE_REF4>(p, scatter, kind, rho, nblocks, list, n, s);
      case RULE_EXACT4: return mass_rule_t<4, RULE_EXACT4>(p, scatter, kind, rho, nblocks, list, n, s);
      case RULE_CENTROID: return mass_rule_t<4, RULE_CENTROID>(p, scatter, kind, rho, nblocks, list, n, s);
      default: return mass_rule_t<4, RULE_REF5>(p, scatter, kind, rho, nblocks, list, n, s);
    }
  }
  switch (rule) {
    case RULE_REF4: return mass_rule_t<10, RULE_REF4>(p, scatter, kind, rho, nblocks, list, n, s);
    case RULE_EXACT4: return mass_rule_t<10, RULE_EXACT4>(p, scatter, kind, rho, nblocks, list, n, s);
    default: return mass_rule_t<10, RULE_REF5>(p, scatter, kind, rho, nblocks, list, n, s);
  }
}

hipError_t launch_elem_dt(const Params &p, double *out, hipStream_t s) {
  const int grid = (p.ne + 255) / 256;
  if (p.npe == 4) CPI_LAUNCH(k_elem_dt<4>, grid, 256, 0, s, p, out);
  CPI_LAUNCH(k_elem_dt<10>, grid, 256, 0, s, p, out);
}

hipError_t launch_import_nodes(const double *src, const int32_t *ninv, int n, Vec3 *d3, Node4 *d4,
                               hipStream_t s) {
  CPI_LAUNCH(k_import_nodes, (unsigned)((3L * n + 255) / 256), 256, 0, s, src, ninv, n, d3, d4);
}

hipError_t launch_export_nodes(const Params &p, const int32_t *ninv, int n, const NodeExport &o,
                               hipStream_t s) {
  CPI_LAUNCH(k_export_nodes, (unsigned)((3L * n + 255) / 256), 256, 0, s, p, ninv, n, o);
}

hipError_t launch_export_elems(const Params &p, int prec, const uint32_t *spos, int n, double *sig,
                               double *ep, hipStream_t s) {
  const unsigned grid = (unsigned)(((long)n * p.nq * (sig ? 6 : 1) + 255) / 256);
  if (prec == 1) CPI_LAUNCH(k_export_elems<float>, grid, 256, 0, s, p, spos, n, sig, ep);
  CPI_LAUNCH(k_export_elems<double>, grid, 256, 0, s, p, spos, n, sig, ep);
}

hipError_t launch_reset_nodes(const Params &p, const Vec3 *v0, hipStream_t s) {
  CPI_LAUNCH(k_reset_nodes, (p.nn + 255) / 256, 256, 0, s, p, v0);
}

hipError_t launch_mass_min(const Params &p, double *out, int blocks, hipStream_t s) {
  CPI_LAUNCH(k_mass_min, blocks, 256, 0, s, (const double *)p.m, p.nn, out);
}

hipError_t launch_stress_node(const Params &p, const int32_t *last, int n, double *strain,
                              double *stress, hipStream_t s) {
  const int grid = (n + 255) / 256;
  if (p.npe == 4) CPI_LAUNCH(k_stress_node<4>, grid, 256, 0, s, p, last, n, strain, stress);
  CPI_LAUNCH(k_stress_node<10>, grid, 256, 0, s, p, last, n, strain, stress);
}

hipError_t launch_debug_strain(const Params &p, int rule, double alpha, int dcase, double nu,
                               double *out, hipStream_t s) {
  const int grid = (p.ne + 255) / 256;
#define CPI_DS(NPE, RULE) \
  CPI_LAUNCH((k_debug_strain<NPE, RULE>), grid, 256, 0, s, p, alpha, dcase, nu, out)
  if (p.npe == 4) {
    switch (rule) {
      case RULE_REF4: CPI_DS(4, RULE_REF4);
      case RULE_EXACT4: CPI_DS(4, RULE_EXACT4);
      case RULE_CENTROID: CPI_DS(4, RULE_CENTROID);
      default: CPI_DS(4, RULE_REF5);
    }
  }
  switch (rule) {
    case RULE_REF4: CPI_DS(10, RULE_REF4);
    case RULE_EXACT4: CPI_DS(10, RULE_EXACT4);
    default: CPI_DS(10, RULE_REF5);
  }
#undef CPI_DS
}

hipError_t launch_mlp_rows(const MlpParams *P, uint16_t *rows, int n, hipStream_t s) {
  if (n <= 0) return hipSuccess;
  const int tiles = (n + 15) / 16;
  const int grid = std::min(kMlpQueueGrid, (tiles + 3) / 4);
  CPI_LAUNCH((k_mlp_queue<kMlpQueueThreads>), grid, kMlpQueueThreads, 0, s, P, rows,
             (const unsigned long long *)nullptr, n);
}

hipError_t launch_stream_copy(const void *src, void *dst, long n4, hipStream_t s) {
  const int grid = (int)std::min<long>((n4 + 255) / 256, 8L * 1024);
  CPI_LAUNCH(k_stream_copy, grid, 256, 0, s, (const Node4 *)src, (Node4 *)dst, n4);
}

}  // namespace cpi
