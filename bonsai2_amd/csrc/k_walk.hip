// k_walk.hip -- computeForces on CDNA4 (reference code/computeForces.cu).
//
// One wave64 per group of <= 64 i-particles (one per lane), pulled from a
// device-wide atomic queue by a persistent grid (the reference's
// retired_groupCount loop, :514-522).  Per group:
//   * the group box is the min/max of its particles (:539-555);
//   * the walk starts at the group's level-1 cells (:259-263) and keeps a
//     per-wave LIFO of cells in global memory (the learned-angle walk keeps
//     its top 1024 entries in LDS); each step pops up to 64 cells,
//     one per lane, and applies the reference's rules: open iff
//     ds^2 < cellOp^2 (:30-54) or the cell holds < 3 particles (:284-285);
//     opened nodes push their children, unopened cells join the P2C list,
//     opened leaves put their particles on the P2P list (:293-430);
//   * lists are kept in LDS, compacted with ballots and prefix sums; every 64
//     entries the wave evaluates the batch.  Two ways to feed the j-data:
//     LDS (default) -- the wave stages the batch (relative to the group
//     centre) in LDS and sweeps it with broadcast ds_read_b128; scalar --
//     the batch index is moved to an SGPR with readlane and the 48-byte cell
//     record (or particle) is fetched by s_load through the scalar cache.
//     Both run at the same rate on MI355X: the FP32 VALU issue rate bounds
//     the walk, not LDS or the scalar cache;
//   * each batch is summed in FP32 and folded into Kahan-compensated
//     accumulators.
// Systems of at most 2^19 particles are walked by the four waves of a block per
// group instead (k_walk_team below).
// The interaction set equals the reference's (the order of traversal does
// not change which cells are opened); FP32 sums run in a different order.
// P2P is code/computeForces.cu:58-78 (20 flops), P2C :83-128 (64 flops),
// rearranged algebraically on a per-cell record with the quadrupole
// pre-scaled and the trace terms precomputed (34 VALU instructions).
#include "bt_device.h"
#include "bt_internal.h"
#include "bt_interact.h"
#include "bt_learn.h"

namespace bt {

namespace {

constexpr int kBlock = 256;
constexpr int kWavesPerBlock = kBlock / kWave;
constexpr int kMaxWalkSteps = 1 << 20;
static_assert(kSafeStack == 8 + kMaxLevel * 448, "entries left behind on every level");

// Unroll of the full-batch j-loops and the occupancy target of the walk.
#ifndef BT_UNROLL_LDS
#define BT_UNROLL_LDS 8
#endif
#ifndef BT_UNROLL_S
#define BT_UNROLL_S 8
#endif
#ifndef BT_UNROLL_LDS2
#define BT_UNROLL_LDS2 4
#endif
#ifndef BT_WALK_WAVES_PER_EU
#define BT_WALK_WAVES_PER_EU 1
#endif
#ifndef BT_LEARN_WAVES_PER_EU
#define BT_LEARN_WAVES_PER_EU 4
#endif
#ifndef BT_LEARN2_WAVES_PER_EU
#define BT_LEARN2_WAVES_PER_EU 3   // two i-particles per lane: 4 would spill VGPRs
#endif
constexpr int kXcd = 8;   // MI355X: 8 XCDs, workgroups dispatched round-robin over them
// Entries of an FP32 walk's stack held in LDS per wave (kLdsStack = 1024,
// 4 KiB).  The FP32 walks run at 4 waves per SIMD (their registers allow no
// more), so 4 blocks of 34 KiB share a CU's 160 KiB of LDS; the FP64 walk
// keeps its whole stack in global memory.  A deeper stack spills its oldest
// entries to the wave's global stack.  The part used (WalkArgs::lstk_cap) is
// at least the 8 * 64 children one step can push, so a step's pushes always
// fit after a spill.

// The groups (PH order) are cut into kXcd contiguous ranges, so neighbouring
// groups share an XCD's L2: range x.
__device__ __forceinline__ int xcd_lo(int ngroups, int x) {
  return (int)((long long)ngroups * x / kXcd);
}
// Next group for this wave: each range has a queue, which a wave drains for its
// own XCD first and then for the others.  Every lane joins the atomics (lane 0
// adds 1) and all branches are uniform.  (Reading a queue's head before adding
// to it, or a fixed first group per wave, measured 1-5% slower at 2^24: 26.8 ms
// as it is, 27.4 and 28.2 ms.)
__device__ __forceinline__ int next_group(DevCounters *dc, int ngroups, int home, int &xr) {
  const int lane = lane_id();
  while (xr < kXcd) {
    const int x = (home + xr) & (kXcd - 1);
    const int lo = xcd_lo(ngroups, x);
    const int k = wave_uniform(atomicAdd(&dc->xq[x], lane == 0 ? 1 : 0));
    if (lo + k < xcd_lo(ngroups, x + 1)) return lo + k;
    xr++;
  }
  return ngroups;
}

// R: the real type of particles, cell data and arithmetic (float for
// Treecode<float>, double for Treecode<double>).
template <typename R>
struct WalkArgs {
  int n, nsys;
  R eps2;
  const int2 *groups;
  const int *group_sys;
  const int2 *root_cells;
  const V4<R> *pos_ph;
  const V4<R> *pos_tree;
  const uint4 *cells;
  const V4<R> *csize;
  const V4<R> *cmono;
  const V4<R> *cq0;
  const V2<R> *cq1;
  const V4<R> *cwalk;    // 3 per cell: (com, M) -7.5(Qxx,Qyy,Qzz,Qxy) (-7.5Qxz,-7.5Qyz,trQ,1.5trQ)
  // learned opening angle (Treecode<float> only)
  const float2 *cls;     // (l, s) per cell
  const float2 *sys_scale;
  const MlpDev *mlp;
  float shift, it_min, it_max;
  V4<R> *acc;
  int2 *gcounts;
  double *gpot;
  int *stack;
  int stack_ints;
  int lstk_cap;          // LDS part of a learned walk's stack, entries per wave
  const int *run_if;     // nullptr, or a device flag: walk only if it is nonzero
  DevCounters *dc;
};

// The i-particles one lane carries.  IPL = 1: particle `lane` of the group.
// IPL = 2: particles 2q and 2q + 1 (q = lane & 31), carried by both halves of
// the wave; each batch of j-entries is split between the half-waves (lanes
// 0-31 sweep its first half, lanes 32-63 its second), so every broadcast LDS
// read serves two interactions, and the halves' sums are added once per group.
//
// A group of np <= 32 particles would leave half of the lanes or more idle: with
// IPL = 1 the wave then holds `slices` copies of the group, lane l particle l % np,
// and copy l / np sweeps the entries copy, copy + slices, ... of each batch.  The
// copies' sums are added once per group, in FP64.  (A group has 28 particles on
// average in a system of 2^16, four in one of 2^10.)  256 systems of 2^10 to 2^16:
// 8.8 -> 7.5 ms per walk.
template <typename R, int IPL>
struct IParts {
  R x[IPL], y[IPL], z[IPL];
  Acc4T<R> s[IPL], c[IPL];   // Kahan sums and compensations
  int slices, slice;         // copies of the group, and this lane's
};

// Copies of a group of np particles: as many as fit, of the numbers whose rounds
// over a batch of 64 entries end within kJSlots slots.
__device__ __forceinline__ int group_slices(int np) {
  const int s = kWave / np;
  return s >= 16 ? 16 : s >= 8 ? 8 : s >= 6 ? 6 : s;
}

// LDS slots of one batch: 64 entries; with IPL = 2 the second half-wave's
// entries start one slot later (its broadcast address differs from the first
// half's by 132 dwords, not a multiple of the bank count) and one zero-mass
// slot follows an odd count.
constexpr int kJSlots = kWave + 2;

template <typename R>
struct Stage {
  V4<R> jA[kJSlots];    // P2C: (com - gc, M)         P2P: (x - gc, m)
  V4<R> jB[kJSlots];    // P2C: -7.5 (Qxx, Qyy, Qzz, Qxy)
  V4<R> jC[kJSlots];    // P2C: (-7.5 Qxz, -7.5 Qyz, trQ, 1.5 trQ)
};

template <typename R>
struct WaveShared : Stage<R> {
  int alist[2 * kWave];
  int dlist[2 * kWave];
  int lpre[kWave];
  int lbeg[kWave];
};

__device__ __forceinline__ float rabs(float v) { return __builtin_fabsf(v); }
__device__ __forceinline__ double rabs(double v) { return __builtin_fabs(v); }

// ds^2 of the improved Barnes-Hut opening test, code/computeForces.cu:30-54
// (same operations in real_t).
template <typename R>
__device__ __forceinline__ R box_ds2(const V4<R> cs, R gcx, R gcy, R gcz, R gsx, R gsy, R gsz) {
#pragma clang fp contract(off)
  R dx = rabs(gcx - cs.x) - gsx;
  R dy = rabs(gcy - cs.y) - gsy;
  R dz = rabs(gcz - cs.z) - gsz;
  dx += rabs(dx); dx *= R(0.5);
  dy += rabs(dy); dy *= R(0.5);
  dz += rabs(dz); dz *= R(0.5);
  return dx * dx + dy * dy + dz * dz;
}

// The test itself: open iff ds^2 < cellOp^2.
template <typename R>
__device__ __forceinline__ bool open_cell(const V4<R> cs, R gcx, R gcy, R gcz, R gsx, R gsy,
                                          R gsz) {
  return box_ds2<R>(cs, gcx, gcy, gcz, gsx, gsy, gsz) < rabs(cs.w);
}

template <bool KAHAN, typename R>
__device__ __forceinline__ void fold(Acc4T<R> &s, Acc4T<R> &c, const Acc4T<R> &b) {
  if (KAHAN) {
    R y, t;
    y = b.x - c.x; t = s.x + y; c.x = (t - s.x) - y; s.x = t;
    y = b.y - c.y; t = s.y + y; c.y = (t - s.y) - y; s.y = t;
    y = b.z - c.z; t = s.z + y; c.z = (t - s.z) - y; s.z = t;
    y = b.w - c.w; t = s.w + y; c.w = (t - s.w) - y; s.w = t;
  } else {
    s.x += b.x; s.y += b.y; s.z += b.z; s.w += b.w;
  }
}

// Entries per half-wave of a batch of cnt, and the LDS slot of entry k.
template <int IPL>
__device__ __forceinline__ int half_count(int cnt) { return IPL == 2 ? (cnt + 1) >> 1 : cnt; }
template <int IPL>
__device__ __forceinline__ int jslot(int k, int hc) { return IPL == 2 ? k + (k >= hc ? 1 : 0) : k; }

// A zero-mass entry far from the group: every term it adds is exactly zero.
template <typename R>
__device__ __forceinline__ void stage_pad(Stage<R> &S, int slot) {
  S.jA[slot] = make_v4<R>(R(1.0e18), R(0), R(0), R(0));
  S.jB[slot] = make_v4<R>(R(0), R(0), R(0), R(0));
  S.jC[slot] = make_v4<R>(R(0), R(0), R(0), R(0));
}

// The slots past a batch of 64 that the copies of a small group may read.
template <typename R>
__device__ __forceinline__ void stage_tail(Stage<R> &S) {
  if (lane_id() < kJSlots - kWave) stage_pad(S, kWave + lane_id());
}

// Whether this lane stages a pad: the copies of a small group sweep cnt entries
// rounded up to a multiple of their number.
template <typename R, int IPL>
__device__ __forceinline__ bool pads(const IParts<R, IPL> &ip, int cnt) {
  const int lane = lane_id();
  if (IPL == 2) return lane == cnt;
  return ip.slices > 1 && lane >= cnt && lane < cnt + ip.slices;
}

// Sweeps a staged batch: P2C (QUAD) or particle-like (P2P and monopole-only
// P2C) interactions of the lane's i-particles with its half of the entries.
template <bool KAHAN, bool QUAD, typename R, int IPL>
__device__ __forceinline__ void sweep(const Stage<R> &S, int cnt, R eps2,
                                      IParts<R, IPL> &ip) {
  const int lane = lane_id();
  Acc4T<R> b[IPL], e[IPL];
#pragma unroll
  for (int k = 0; k < IPL; k++) b[k] = e[k] = Acc4T<R>{R(0), R(0), R(0), R(0)};
  // One entry's j-data, and its interactions with the lane's i-particles.
  struct J {
    V4<R> A, B, C;
  };
  auto load = [&](int slot) {
    J j;
    j.A = S.jA[slot];
    if (QUAD) {
      j.B = S.jB[slot];
      j.C = S.jC[slot];
    }
    return j;
  };
  auto eval = [&](const J &j) {
    if (QUAD) {
#pragma unroll
      for (int k = 0; k < IPL; k++)
        p2c_rec(b[k], e[k], ip.x[k], ip.y[k], ip.z[k], j.A, j.B, j.C, eps2);
    } else {
#pragma unroll
      for (int k = 0; k < IPL; k++) p2p(b[k], ip.x[k], ip.y[k], ip.z[k], j.A, eps2);
    }
  };
  // Entry j + 1 is read from LDS while entry j is evaluated, so the reads'
  // latency is hidden behind one interaction's arithmetic.  The read past the
  // last entry stays inside the kJSlots slots and its value is not used.
  if (IPL == 2) {
    const int hc = half_count<2>(cnt);
    const int base = lane >= 32 ? hc + 1 : 0;
    J cur = load(base);
    if (cnt == kWave) {
#pragma unroll BT_UNROLL_LDS2
      for (int j = 0; j < kWave / 2; j++) {
        const J nxt = load(base + j + 1);
        __builtin_amdgcn_sched_barrier(0);   // keep the reads ahead of the arithmetic
        eval(cur);
        cur = nxt;
      }
    } else {
#pragma unroll 2
      for (int j = 0; j < hc; j++) {
        const J nxt = load(base + j + 1);
        __builtin_amdgcn_sched_barrier(0);   // keep the reads ahead of the arithmetic
        eval(cur);
        cur = nxt;
      }
    }
  } else if (ip.slices > 1) {
    const int rounds = (cnt + ip.slices - 1) / ip.slices;
    int slot = ip.slice;
    J cur = load(slot);
#pragma unroll 2
    for (int j = 1; j <= rounds; j++) {
      slot += j < rounds ? ip.slices : 0;
      const J nxt = load(slot);
      __builtin_amdgcn_sched_barrier(0);   // keep the reads ahead of the arithmetic
      eval(cur);
      cur = nxt;
    }
  } else {
    J cur = load(0);
    if (cnt == kWave) {
#pragma unroll BT_UNROLL_LDS
      for (int j = 0; j < kWave; j++) {
        const J nxt = load(j + 1);
        __builtin_amdgcn_sched_barrier(0);   // keep the reads ahead of the arithmetic
        eval(cur);
        cur = nxt;
      }
    } else {
#pragma unroll 2
      for (int j = 0; j < cnt; j++) {
        const J nxt = load(j + 1);
        __builtin_amdgcn_sched_barrier(0);   // keep the reads ahead of the arithmetic
        eval(cur);
        cur = nxt;
      }
    }
  }
#pragma unroll
  for (int k = 0; k < IPL; k++) {
    if (QUAD) p2c_finish(b[k], e[k]);
    fold<KAHAN, R>(ip.s[k], ip.c[k], b[k]);
  }
}

template <bool KAHAN, typename R, int IPL>
__device__ __forceinline__ void eval_p2c(const WalkArgs<R> &a, Stage<R> &S, const int *list, int cnt, R gcx,
                                         R gcy, R gcz, IParts<R, IPL> &ip) {
  const int lane = lane_id();
  const int hc = half_count<IPL>(cnt);
  if (lane < cnt) {
    const int ci = list[lane];
    const V4<R> r0 = a.cwalk[3 * ci];
    const int d = jslot<IPL>(lane, hc);
    S.jA[d] = make_v4<R>(r0.x - gcx, r0.y - gcy, r0.z - gcz, r0.w);
    S.jB[d] = a.cwalk[3 * ci + 1];
    S.jC[d] = a.cwalk[3 * ci + 2];
  } else if (pads<R, IPL>(ip, cnt)) {
    stage_pad(S, IPL == 2 ? cnt + 1 : lane);
  }
  wave_lds_sync();
  sweep<KAHAN, true, R, IPL>(S, cnt, a.eps2, ip);
  wave_lds_sync();
}

template <bool KAHAN, typename R, int IPL>
__device__ __forceinline__ void eval_p2p(const WalkArgs<R> &a, Stage<R> &S, const int *list, int cnt, R gcx,
                                         R gcy, R gcz, IParts<R, IPL> &ip) {
  const int lane = lane_id();
  const int hc = half_count<IPL>(cnt);
  if (lane < cnt) {
    const V4<R> p = a.pos_tree[list[lane]];
    S.jA[jslot<IPL>(lane, hc)] = make_v4<R>(p.x - gcx, p.y - gcy, p.z - gcz, p.w);
  } else if (pads<R, IPL>(ip, cnt)) {
    stage_pad(S, IPL == 2 ? cnt + 1 : lane);
  }
  wave_lds_sync();
  sweep<KAHAN, false, R, IPL>(S, cnt, a.eps2, ip);
  wave_lds_sync();
}

// Monopole-only P2C (the reference built without QUADRUPOLE,
// code/computeForces.cu:198-225): the cell's mass at its centre of mass,
// evaluated like a particle (20 flops).
template <bool KAHAN, typename R, int IPL>
__device__ __forceinline__ void eval_p2c_mono(const WalkArgs<R> &a, Stage<R> &S, const int *list, int cnt,
                                              R gcx, R gcy, R gcz, IParts<R, IPL> &ip) {
  const int lane = lane_id();
  const int hc = half_count<IPL>(cnt);
  if (lane < cnt) {
    const V4<R> r0 = a.cwalk[3 * list[lane]];
    S.jA[jslot<IPL>(lane, hc)] = make_v4<R>(r0.x - gcx, r0.y - gcy, r0.z - gcz, r0.w);
  } else if (pads<R, IPL>(ip, cnt)) {
    stage_pad(S, IPL == 2 ? cnt + 1 : lane);
  }
  wave_lds_sync();
  sweep<KAHAN, false, R, IPL>(S, cnt, a.eps2, ip);
  wave_lds_sync();
}

// Cell records and particles do not change during the walk: reading them
// through the constant address space lets the compiler fetch a wave-uniform
// record with s_load (scalar cache) instead of a vector load.
typedef float f4v __attribute__((ext_vector_type(4)));
typedef __attribute__((address_space(4))) const f4v cf4v;

__device__ __forceinline__ float4 ld_uniform(const cf4v *p, int i) {
  const f4v v = p[i];
  return make_float4(v[0], v[1], v[2], v[3]);
}

// Scalar-load j-data (one i-particle per lane, absolute coordinates).
template <bool KAHAN>
__device__ __forceinline__ void eval_p2c_s(const WalkArgs<float> &a, const int *list,
                                           int cnt, IParts<float, 1> &ip) {
  const cf4v *rec = (const cf4v *)a.cwalk;
  const int my = list[lane_id()];
  Acc4 b = {0.f, 0.f, 0.f, 0.f}, e = b;
  if (cnt == kWave) {
#pragma unroll BT_UNROLL_S
    for (int j = 0; j < kWave; j++) {
      const int r = 3 * __builtin_amdgcn_readlane(my, j);
      p2c_rec(b, e, ip.x[0], ip.y[0], ip.z[0], ld_uniform(rec, r), ld_uniform(rec, r + 1),
              ld_uniform(rec, r + 2), a.eps2);
    }
  } else {
#pragma unroll 2
    for (int j = 0; j < cnt; j++) {
      const int r = 3 * __builtin_amdgcn_readlane(my, j);
      p2c_rec(b, e, ip.x[0], ip.y[0], ip.z[0], ld_uniform(rec, r), ld_uniform(rec, r + 1),
              ld_uniform(rec, r + 2), a.eps2);
    }
  }
  p2c_finish(b, e);
  fold<KAHAN>(ip.s[0], ip.c[0], b);
}

template <bool KAHAN>
__device__ __forceinline__ void eval_p2p_s(const WalkArgs<float> &a, const int *list,
                                           int cnt, IParts<float, 1> &ip) {
  const cf4v *pj = (const cf4v *)a.pos_tree;
  const int my = list[lane_id()];
  Acc4 b = {0.f, 0.f, 0.f, 0.f};
  if (cnt == kWave) {
#pragma unroll BT_UNROLL_S
    for (int j = 0; j < kWave; j++)
      p2p(b, ip.x[0], ip.y[0], ip.z[0], ld_uniform(pj, __builtin_amdgcn_readlane(my, j)), a.eps2);
  } else {
#pragma unroll 2
    for (int j = 0; j < cnt; j++)
      p2p(b, ip.x[0], ip.y[0], ip.z[0], ld_uniform(pj, __builtin_amdgcn_readlane(my, j)), a.eps2);
  }
  fold<KAHAN>(ip.s[0], ip.c[0], b);
}

// One batch of cnt P2C (list of cells) or P2P (list of particles) interactions.  The
// LDS path takes i relative to the group centre, the scalar path absolute i.
template <bool KAHAN, bool SJ, bool MONO, typename R, int IPL>
__device__ __forceinline__ void batch_p2c(const WalkArgs<R> &a, Stage<R> &S, const int *list, int cnt, R gcx,
                                          R gcy, R gcz, IParts<R, IPL> &ip) {
  if constexpr (MONO) eval_p2c_mono<KAHAN, R, IPL>(a, S, list, cnt, gcx, gcy, gcz, ip);
  else if constexpr (SJ) eval_p2c_s<KAHAN>(a, list, cnt, ip);
  else eval_p2c<KAHAN, R, IPL>(a, S, list, cnt, gcx, gcy, gcz, ip);
}

template <bool KAHAN, bool SJ, typename R, int IPL>
__device__ __forceinline__ void batch_p2p(const WalkArgs<R> &a, Stage<R> &S, const int *list, int cnt, R gcx,
                                          R gcy, R gcz, IParts<R, IPL> &ip) {
  if constexpr (SJ) eval_p2p_s<KAHAN>(a, list, cnt, ip);
  else eval_p2p<KAHAN, R, IPL>(a, S, list, cnt, gcx, gcy, gcz, ip);
}

// The network's operands of one wave: matrix-core operands in registers, bias
// and output rows in the block's LDS (64 floats).
struct Net {
  half8_t a1, a2_0, a2_1;
  float b3;
  const float *s_mlp;
  // all threads of the block
  __device__ __forceinline__ void load(const MlpDev *m, float *s) {
    const int t = threadIdx.x, lane = lane_id();
    if (t < 32) s[t] = m->c2p[t >> 4][t & 15];
    else if (t < 64) s[t] = m->w3p[(t - 32) >> 4][t & 15];
    a1 = m->a1[lane];
    a2_0 = m->a2[0][lane];
    a2_1 = m->a2[1][lane];
    b3 = m->b3;
    s_mlp = s;
    __syncthreads();
  }
};

// Whether this lane's cell is opened for the group (all lanes of the wave call;
// `use`: the lane has a cell).  LEARN: by the network's angle for the pair.
template <typename R, bool LEARN>
__device__ __forceinline__ bool opens(const WalkArgs<R> &a, bool use, int ci, const uint4 cd,
                                      const V4<R> cs, R gcx, R gcy, R gcz, R gsx, R gsy, R gsz,
                                      const GroupGeom &geom, const Net &net) {
  if constexpr (LEARN) {
  float2 lsv = make_float2(0.f, 0.f);
    if (use) lsv = a.cls[ci];
    // A cell opened even at theta_hi or accepted even at theta_lo is
    // decided without the network: (l/theta + s)^2 is monotone in 1/theta,
    // so every angle of the band gives it the same answer.  Only a step
    // with an undecided cell loads the moments and computes features, and
    // only a 32-lane block holding one evaluates the network.
    const float ds2 = box_ds2(cs, gcx, gcy, gcz, gsx, gsy, gsz);
    float op_lo, op_hi;
    {
#pragma clang fp contract(off)
      op_lo = lsv.x * a.it_max + lsv.y;
      op_hi = lsv.x * a.it_min + lsv.y;
      op_lo = op_lo * op_lo;
      op_hi = op_hi * op_hi;
    }
    const bool undecided = use && ds2 < op_lo && ds2 >= op_hi;
    const uint64_t um = ballot64(undecided);
    float it = a.it_min;
    if (um != 0) {
      // every lane evaluates the network (decided and idle lanes on a zero cell)
      float4 m = make_float4(0.f, 0.f, 0.f, 0.f), q0 = m;
      float2 q1 = make_float2(0.f, 0.f);
      if (undecided) {
        m = a.cmono[ci];
        q0 = a.cq0[ci];
        q1 = a.cq1[ci];
      }
      float x[8];
      pair_features(geom, m, lsv.x, q0, q1, x);
      const float y = mlp_wave(net.a1, net.a2_0, net.a2_1, net.s_mlp, net.b3, pack_features(x),
                               (um & 0xFFFFFFFFull) != 0, (um >> 32) != 0);
      it = learned_inv_theta(y, a.shift, a.it_min, a.it_max);
    }
    float op;
    {
#pragma clang fp contract(off)
      op = lsv.x * it + lsv.y;
      op = op * op;
    }
    // the opening test of open_cell with this pair's radius (same ds^2)
    return use && (ds2 < op || ((int)cd.w - (int)cd.z < 3));
  } else {
    return use && (open_cell<R>(cs, gcx, gcy, gcz, gsx, gsy, gsz) || ((int)cd.w - (int)cd.z < 3));
  }
}

// LEARN: each popped cell gets its own opening angle from the network
// (bt_learn.h), evaluated by the wave on the matrix cores for up to 64 cells.
// MONO: monopole-only P2C (the reference's build without QUADRUPOLE).
template <typename R, bool KAHAN, bool SJ, bool LEARN, bool MONO, int IPL>
__global__ __launch_bounds__(kBlock)
__attribute__((amdgpu_waves_per_eu(LEARN ? (IPL == 2 ? BT_LEARN2_WAVES_PER_EU : BT_LEARN_WAVES_PER_EU)
                                         : BT_WALK_WAVES_PER_EU)))
void k_walk(WalkArgs<R> a) {
  static_assert(!(LEARN || SJ) || sizeof(R) == 4, "learned angle and scalar loads: FP32 only");
  __shared__ WaveShared<R> sh[kWavesPerBlock];
  __shared__ float s_mlp[LEARN ? 64 : 1];
  constexpr bool LSTK = sizeof(R) == 4;
  __shared__ int s_stack[LSTK ? kWavesPerBlock * kLdsStack : 1];
  const int lane = lane_id();
  const int wv = threadIdx.x >> 6;
  WaveShared<R> &S = sh[wv];
  // LSTK: the top of the stack (up to kLdsStack entries) lives in LDS, the
  // older entries below it in global memory (stk[0, gtop)); otherwise the
  // whole stack is in global memory (stk[0, top))
  int *stk = a.stack + (size_t)(blockIdx.x * kWavesPerBlock + wv) * (size_t)a.stack_ints;
  int *lstk = s_stack + (LSTK ? wv * kLdsStack : 0);
  Net net;
  if constexpr (LEARN) net.load(a.mlp, s_mlp);
  if (a.run_if && *a.run_if == 0) return;   // a fallback walk that is not needed
  const int ngroups = a.dc->ngroups;
  // a failed build (cell or group capacity) leaves placeholder links: do not walk it
  if (a.dc->err & (3 | kSortErr | kShortErr)) return;

  // The persistent loop has no lane-dependent branches at its ends: two
  // "if (lane == 0)" blocks around the back edge (queue fetch, stats store) are
  // merged by the compiler into a region that only lane 0 re-enters, leaving
  // the other lanes to loop on a stale group index.  Every lane therefore
  // joins the queue atomic (lane 0 adds 1, the others 0) and the per-group
  // stores below are branch-free.
  const int home = (int)(blockIdx.x % kXcd);
  int xr = 0;
  for (;;) {
    const int g = next_group(a.dc, ngroups, home, xr);
    if (g >= ngroups) break;
    const int2 grp = a.groups[g];
    const int pbeg = grp.x, np = max(grp.y, 1);
    const int sys = a.nsys > 1 ? a.group_sys[g] : 0;
    const int slices = IPL == 1 && !SJ ? group_slices(np) : 1;
    // the lane's i-particles (clamped to the last one, :534)
    V4<R> pi[IPL];
#pragma unroll
    for (int k = 0; k < IPL; k++)
      pi[k] = a.pos_ph[pbeg + (IPL == 1 ? (slices > 1 ? lane % np : min(lane, np - 1))
                                        : min(2 * (lane & 31) + k, np - 1))];

    // group box (code/computeForces.cu:539-555)
    R lmnx = pi[0].x, lmny = pi[0].y, lmnz = pi[0].z;
    R lmxx = pi[0].x, lmxy = pi[0].y, lmxz = pi[0].z;
#pragma unroll
    for (int k = 1; k < IPL; k++) {
      lmnx = rmin(lmnx, pi[k].x); lmny = rmin(lmny, pi[k].y); lmnz = rmin(lmnz, pi[k].z);
      lmxx = rmax(lmxx, pi[k].x); lmxy = rmax(lmxy, pi[k].y); lmxz = rmax(lmxz, pi[k].z);
    }
    const R mnx = wave_min_r(lmnx), mny = wave_min_r(lmny), mnz = wave_min_r(lmnz);
    const R mxx = wave_max_r(lmxx), mxy = wave_max_r(lmxy), mxz = wave_max_r(lmxz);
    R gcx, gcy, gcz, gsx, gsy, gsz;
    {
#pragma clang fp contract(off)
      gcx = R(0.5) * (mxx + mnx); gcy = R(0.5) * (mxy + mny); gcz = R(0.5) * (mxz + mnz);
      gsx = R(0.5) * (mxx - mnx); gsy = R(0.5) * (mxy - mny); gsz = R(0.5) * (mxz - mnz);
    }
    GroupGeom geom;
    if constexpr (LEARN) geom = make_group_geom(gcx, gcy, gcz, gsx, gsy, gsz, np, a.sys_scale[sys]);
    // i-particles: relative to the group centre (LDS path) or absolute (scalar path)
    IParts<R, IPL> ip;
    ip.slices = slices;
    ip.slice = min(lane / np, slices - 1);
    if (IPL == 1) stage_tail(S);
#pragma unroll
    for (int k = 0; k < IPL; k++) {
      ip.x[k] = SJ ? pi[k].x : pi[k].x - gcx;
      ip.y[k] = SJ ? pi[k].y : pi[k].y - gcy;
      ip.z[k] = SJ ? pi[k].z : pi[k].z - gcz;
      ip.s[k] = Acc4T<R>{R(0), R(0), R(0), R(0)};
      ip.c[k] = Acc4T<R>{R(0), R(0), R(0), R(0)};
    }

    const int2 rc = a.root_cells[sys];
    if (lane < rc.y) {
      if (LSTK) lstk[lane] = rc.x + lane;
      else stk[lane] = rc.x + lane;
    }
    int top = rc.y;
    int gtop = 0;                // LSTK: entries spilled to global memory
    int na = 0, nd = 0;          // pending list lengths
    int n_app = 0, n_dir = 0;    // interactions evaluated (stats)
    int deepest = top;           // stack high-water mark of this group
    bool overflow = false;
    int steps = 0;
    __builtin_amdgcn_s_waitcnt(0);

    while (top > 0 || gtop > 0) {
      // every cell is visited at most once per group; a longer walk means a
      // corrupt tree, so stop rather than loop
      if (++steps > kMaxWalkSteps) {
        overflow = true;
        break;
      }
      if (LSTK && top < kWave && gtop > 0) {
        // top the LDS part up with the newest spilled entries (slid in below
        // the ones left), so that the step pops the same cells as it would
        // from one stack
        const int r = min(gtop, a.lstk_cap / 2);
        const int v = lane < top ? lstk[lane] : 0;
        wave_lds_sync();
        if (lane < top) lstk[r + lane] = v;
        for (int k = lane; k < r; k += kWave) lstk[k] = stk[gtop - r + k];
        gtop -= r;
        top += r;
        wave_lds_sync();
      }
      const int take = min(kWave, top);
      top -= take;
      const bool use = lane < take;
      int ci = 0;
      uint4 cd = make_uint4(0, 0, 0, 0);
      V4<R> cs = make_v4<R>(R(0), R(0), R(0), R(0));
      if (use) {
        ci = LSTK ? lstk[top + lane] : stk[top + lane];
        cd = a.cells[ci];
        cs = a.csize[ci];
      }
      const bool split = opens<R, LEARN>(a, use, ci, cd, cs, gcx, gcy, gcz, gsx, gsy, gsz, geom, net);
      const bool leaf = cell_leaf(cd);
      const bool push = use && split && !leaf;
      const bool approx = use && !split;
      const bool direct = use && split && leaf;

      // children of opened nodes go on the stack
      const int nch = push ? cell_nchild(cd) : 0;
      const int chi = wave_incl_scan(nch);
      const int ctot = last_lane(chi);
      if (LSTK && top + ctot > a.lstk_cap) {
        // spill the oldest LDS entries to the global stack, leaving a quarter
        // of the LDS part free after this step's pushes where possible
        const int sp = min(top, top + ctot - a.lstk_cap + a.lstk_cap / 4);
        if (top - sp + ctot > a.lstk_cap || gtop + sp > a.stack_ints) {
          overflow = true;
          break;
        }
        for (int k = lane; k < sp; k += kWave) stk[gtop + k] = lstk[k];
        wave_lds_sync();
        // move the rest down; each chunk is read in full before it is written
        for (int k0 = 0; k0 < top - sp; k0 += kWave) {
          const int k = k0 + lane;
          const int v = k < top - sp ? lstk[sp + k] : 0;
          wave_lds_sync();
          if (k < top - sp) lstk[k] = v;
          wave_lds_sync();
        }
        gtop += sp;
        top -= sp;
      } else if (!LSTK && top + ctot > a.stack_ints) {
        overflow = true;
        break;
      }
      if (push) {
        const int f = cell_first(cd);
        const int base = top + chi - nch;
        for (int k = 0; k < nch; k++) {
          if (LSTK) lstk[base + k] = f + k;
          else stk[base + k] = f + k;
        }
      }
      top += ctot;
      deepest = max(deepest, top + gtop);

      // approximate list (P2C)
      const uint64_t am = ballot64(approx);
      if (approx) S.alist[na + __popcll(am & lanemask_lt())] = ci;
      na += __popcll(am);

      // direct list (P2P): expand the opened leaves' particle ranges
      const uint64_t dm = ballot64(direct);
      const int ndl = __popcll(dm);
      if (ndl > 0) {
        const int lsz = direct ? (int)cd.w - (int)cd.z : 0;
        const int li = wave_incl_scan(lsz);
        const int ltot = last_lane(li);
        if (direct) {
          const int r = __popcll(dm & lanemask_lt());
          S.lpre[r] = li - lsz;
          S.lbeg[r] = (int)cd.z;
        }
        wave_lds_sync();
        for (int k0 = 0; k0 < ltot; k0 += kWave) {
          const int k = k0 + lane;
          if (k < ltot) {
            int lo = 0, hi = ndl - 1;  // last leaf with lpre <= k
            while (lo < hi) {
              const int mid = (lo + hi + 1) >> 1;
              if (S.lpre[mid] <= k) lo = mid; else hi = mid - 1;
            }
            S.dlist[nd + lane] = S.lbeg[lo] + (k - S.lpre[lo]);
          }
          nd += min(kWave, ltot - k0);
          wave_lds_sync();
          if (nd >= kWave) {
            batch_p2p<KAHAN, SJ, R, IPL>(a, S, S.dlist, kWave, gcx, gcy, gcz, ip);
            n_dir += kWave;
            nd -= kWave;
            if (lane < nd) S.dlist[lane] = S.dlist[kWave + lane];
            wave_lds_sync();
          }
        }
      }
      wave_lds_sync();
      if (na >= kWave) {
        batch_p2c<KAHAN, SJ, MONO, R, IPL>(a, S, S.alist, kWave, gcx, gcy, gcz, ip);
        n_app += kWave;
        na -= kWave;
        if (lane < na) S.alist[lane] = S.alist[kWave + lane];
        wave_lds_sync();
      }
      // stack pushes of this step (stores by some lanes) must have completed
      // before the next step's pops (loads by other lanes)
      __builtin_amdgcn_s_waitcnt(0);
    }
    if (overflow) {
      atomicOr(&a.dc->err, 4);  // every lane, same bit
      atomicOr(&a.dc->err_sticky, 4);
      na = 0;
      nd = 0;
    }
    if (na > 0) {
      batch_p2c<KAHAN, SJ, MONO, R, IPL>(a, S, S.alist, na, gcx, gcy, gcz, ip);
      n_app += na;
    }
    if (nd > 0) {
      batch_p2p<KAHAN, SJ, R, IPL>(a, S, S.dlist, nd, gcx, gcy, gcz, ip);
      n_dir += nd;
    }
    // this lane stores particle `idx`; lanes past the end of the group write
    // to the kWave spare slots after acc[n)
    Acc4T<R> res;
    R mi;
    int idx;
    if (IPL == 1) {
      res = ip.s[0];
      if (slices > 1) {
        // the copies' compensated sums, in their order
        const Acc4T<R> cc = ip.c[0];
        const double v[4] = {(double)res.x - (KAHAN ? (double)cc.x : 0.0),
                             (double)res.y - (KAHAN ? (double)cc.y : 0.0),
                             (double)res.z - (KAHAN ? (double)cc.z : 0.0),
                             (double)res.w - (KAHAN ? (double)cc.w : 0.0)};
        double t[4] = {v[0], v[1], v[2], v[3]};
        for (int k = 1; k < slices; k++)
          for (int q = 0; q < 4; q++) t[q] += __shfl(v[q], lane + k * np, kWave);
        res = Acc4T<R>{(R)t[0], (R)t[1], (R)t[2], (R)t[3]};
      }
      mi = pi[0].w;
      idx = lane;
    } else {
      // each half-wave summed half of every batch: add the other half's sums
      // (compensated values s - c) to get the particles' totals
      const int h = lane >> 5;
      Acc4T<R> t[IPL];
#pragma unroll
      for (int k = 0; k < IPL; k++) {
        Acc4T<R> v = ip.s[k];
        if (KAHAN) {
          v.x -= ip.c[k].x; v.y -= ip.c[k].y; v.z -= ip.c[k].z; v.w -= ip.c[k].w;
        }
        t[k].x = v.x + __shfl_xor(v.x, 32, kWave);
        t[k].y = v.y + __shfl_xor(v.y, 32, kWave);
        t[k].z = v.z + __shfl_xor(v.z, 32, kWave);
        t[k].w = v.w + __shfl_xor(v.w, 32, kWave);
      }
      res = h ? t[IPL - 1] : t[0];
      mi = h ? pi[IPL - 1].w : pi[0].w;
      idx = 2 * (lane & 31) + h;
    }
    const bool valid = idx < np;
    a.acc[valid ? pbeg + idx : a.n + lane] = make_v4<R>(res.x, res.y, res.z, res.w);
    const double gp = wave_sum(valid ? (double)mi * (double)res.w : 0.0);
    a.gcounts[g] = overflow ? make_int2(-1, -1) : make_int2(n_app, n_dir);
    a.gpot[g] = gp;
    atomicMax(&a.dc->stack_max, lane == 0 ? deepest : 0);
    atomicMax(&a.dc->stack_hw, lane == 0 ? deepest : 0);
  }
}

// ---- team walk ----------------------------------------------------------------
//
// With fewer groups than the chip has wave slots, the walk above lasts as long as
// one wave needs for its whole group: it is bound by that wave's dependent loads
// and by one wave's issue rate (one VALU instruction in 6-7 cycles, a SIMD takes
// one in 2.8 from three waves).  Here the T waves of a block walk one group
// together: a step pops up to 64 T cells from one stack in LDS, wave w lane l
// testing the (l T + w)-th from the top's start, so siblings go to different
// waves; children, accepted cells and opened leaves go to shared lists at offsets
// from the waves' counts, and a list of 64 T entries is evaluated as T batches,
// one per wave, each lane holding the same i-particle in all waves.  At the end
// the waves share the rest of both lists out evenly and their compensated sums
// are added in FP64.  The interaction set is that of the walk above.
constexpr int kTeam = kWavesPerBlock;

template <typename R>
struct TeamShared {
  static constexpr int T = kTeam;
  static constexpr int W = T * kWave;       // cells a step pops, entries a round evaluates
  static constexpr int kStack = T * 512;    // holds the 8 W children one step can push
  union {
    Stage<R> stage[T];
    double sum[T][4][kWave];                // after the group's last batch
  };
  int stack[kStack];
  int alist[2 * W], dlist[2 * W];
  int lpre[W], lbeg[W];
  int4 tot[T];
  __device__ TeamShared() {}
};

// All threads of the block, which all see the same counts: takes the first W
// entries off a list of cnt >= W.
template <int W>
__device__ __forceinline__ void drop_round(int *list, int &cnt) {
  __syncthreads();   // every wave has read its entries
  cnt -= W;
  const int t = threadIdx.x;
  if (t < cnt) list[t] = list[W + t];
  __syncthreads();
}

template <typename R, bool KAHAN, bool LEARN, bool MONO>
__global__ __launch_bounds__(kBlock)
__attribute__((amdgpu_waves_per_eu(LEARN ? BT_LEARN_WAVES_PER_EU : BT_WALK_WAVES_PER_EU)))
void k_walk_team(WalkArgs<R> a) {
  typedef TeamShared<R> Sh;
  constexpr int T = kTeam, W = Sh::W, kStack = Sh::kStack;
  __shared__ Sh sh;
  __shared__ float s_mlp[LEARN ? 64 : 1];
  const int lane = lane_id();
  const int wv = wave_uniform((int)(threadIdx.x >> 6));
  const int tid = threadIdx.x;
  Stage<R> &S = sh.stage[wv];
  int *spill = a.stack + (size_t)blockIdx.x * T * (size_t)a.stack_ints;
  const int spill_cap = T * a.stack_ints;
  Net net;
  if constexpr (LEARN) net.load(a.mlp, s_mlp);
  if (a.run_if && *a.run_if == 0) return;
  const int ngroups = a.dc->ngroups;
  if (a.dc->err & (3 | kSortErr | kShortErr)) return;

  // the block's groups: a fixed stride over all of them, so that the groups of a
  // dense region, neighbours in PH order with the longest lists, go to all XCDs (a
  // small system's tree fits every L2).  Every branch below is uniform over the block.
  for (int g = (int)blockIdx.x; g < ngroups; g += (int)gridDim.x) {
    const int2 grp = a.groups[g];
    const int pbeg = grp.x, np = max(grp.y, 1);
    const int sys = a.nsys > 1 ? a.group_sys[g] : 0;
    const int slices = group_slices(np);
    const V4<R> pi = a.pos_ph[pbeg + (slices > 1 ? lane % np : min(lane, np - 1))];
    const R mnx = wave_min_r(pi.x), mny = wave_min_r(pi.y), mnz = wave_min_r(pi.z);
    const R mxx = wave_max_r(pi.x), mxy = wave_max_r(pi.y), mxz = wave_max_r(pi.z);
    R gcx, gcy, gcz, gsx, gsy, gsz;
    {
#pragma clang fp contract(off)
      gcx = R(0.5) * (mxx + mnx); gcy = R(0.5) * (mxy + mny); gcz = R(0.5) * (mxz + mnz);
      gsx = R(0.5) * (mxx - mnx); gsy = R(0.5) * (mxy - mny); gsz = R(0.5) * (mxz - mnz);
    }
    GroupGeom geom;
    if constexpr (LEARN) geom = make_group_geom(gcx, gcy, gcz, gsx, gsy, gsz, np, a.sys_scale[sys]);
    IParts<R, 1> ip;
    ip.slices = slices;
    ip.slice = min(lane / np, slices - 1);
    stage_tail(S);
    ip.x[0] = pi.x - gcx;
    ip.y[0] = pi.y - gcy;
    ip.z[0] = pi.z - gcz;
    ip.s[0] = Acc4T<R>{R(0), R(0), R(0), R(0)};
    ip.c[0] = Acc4T<R>{R(0), R(0), R(0), R(0)};

    const int2 rc = a.root_cells[sys];
    if (tid < rc.y) sh.stack[tid] = rc.x + tid;
    int top = rc.y, gtop = 0;    // entries in LDS, older ones in the spill area
    int na = 0, nd = 0;          // pending list lengths
    int n_app = 0, n_dir = 0;    // interactions evaluated (stats)
    int deepest = top;
    bool overflow = false;
    int steps = 0;
    __syncthreads();

    while (top > 0 || gtop > 0) {
      if (++steps > kMaxWalkSteps) {
        overflow = true;
        break;
      }
      if (top < W && gtop > 0) {
        // the newest spilled entries slide in below the ones left
        const int r = min(gtop, kStack / 2);
        const int v = tid < top ? sh.stack[tid] : 0;
        __syncthreads();
        if (tid < top) sh.stack[r + tid] = v;
        for (int k = tid; k < r; k += W) sh.stack[k] = spill[gtop - r + k];
        gtop -= r;
        top += r;
        __syncthreads();
      }
      const int take = min(W, top);
      top -= take;
      const int e = lane * T + wv;
      const bool use = e < take;
      int ci = 0;
      uint4 cd = make_uint4(0, 0, 0, 0);
      V4<R> cs = make_v4<R>(R(0), R(0), R(0), R(0));
      if (use) {
        ci = sh.stack[top + e];
        cd = a.cells[ci];
        cs = a.csize[ci];
      }
      const bool split = opens<R, LEARN>(a, use, ci, cd, cs, gcx, gcy, gcz, gsx, gsy, gsz, geom, net);
      const bool leaf = cell_leaf(cd);
      const bool push = split && !leaf;
      const bool approx = use && !split;
      const bool direct = split && leaf;
      const int nch = push ? cell_nchild(cd) : 0;
      const int lsz = direct ? (int)cd.w - (int)cd.z : 0;
      const int chi = wave_incl_scan(nch);
      const int li = wave_incl_scan(lsz);
      const uint64_t am = ballot64(approx), dm = ballot64(direct);
      // this wave's counts (the same values from its last lane)
      if (lane == kWave - 1) sh.tot[wv] = make_int4(chi, __popcll(am), __popcll(dm), li);
      __syncthreads();
      int4 before = make_int4(0, 0, 0, 0), all = before;
#pragma unroll
      for (int w = 0; w < T; w++) {
        const int4 t = sh.tot[w];
        if (w < wv) { before.x += t.x; before.y += t.y; before.z += t.z; before.w += t.w; }
        all.x += t.x; all.y += t.y; all.z += t.z; all.w += t.w;
      }
      if (top + all.x > kStack) {
        // the oldest entries leave for the spill area, a quarter stays free
        const int sp = min(top, top + all.x - kStack + kStack / 4);
        if (top - sp + all.x > kStack || gtop + sp > spill_cap) {
          overflow = true;
          break;
        }
        for (int k = tid; k < sp; k += W) spill[gtop + k] = sh.stack[k];
        __syncthreads();
        for (int k0 = 0; k0 < top - sp; k0 += W) {   // each chunk is read before it is written
          const int k = k0 + tid;
          const int v = k < top - sp ? sh.stack[sp + k] : 0;
          __syncthreads();
          if (k < top - sp) sh.stack[k] = v;
          __syncthreads();
        }
        gtop += sp;
        top -= sp;
      }
      if (push) {
        const int f = cell_first(cd);
        const int base = top + before.x + chi - nch;
        for (int k = 0; k < nch; k++) sh.stack[base + k] = f + k;
      }
      if (approx) sh.alist[na + before.y + __popcll(am & lanemask_lt())] = ci;
      if (direct) {
        const int r = before.z + __popcll(dm & lanemask_lt());
        sh.lpre[r] = before.w + li - lsz;
        sh.lbeg[r] = (int)cd.z;
      }
      top += all.x;
      na += all.y;
      deepest = max(deepest, top + gtop);
      __syncthreads();
      // expand the opened leaves' particle ranges, W at a time
      for (int k0 = 0; k0 < all.w; k0 += W) {
        const int k = k0 + tid;
        if (k < all.w) {
          int lo = 0, hi = all.z - 1;  // last leaf with lpre <= k
          while (lo < hi) {
            const int mid = (lo + hi + 1) >> 1;
            if (sh.lpre[mid] <= k) lo = mid; else hi = mid - 1;
          }
          sh.dlist[nd + tid] = sh.lbeg[lo] + (k - sh.lpre[lo]);
        }
        nd += min(W, all.w - k0);
        __syncthreads();
        if (nd >= W) {
          batch_p2p<KAHAN, false, R, 1>(a, S, sh.dlist + wv * kWave, kWave, gcx, gcy, gcz, ip);
          n_dir += W;
          drop_round<W>(sh.dlist, nd);
        }
      }
      if (na >= W) {
        batch_p2c<KAHAN, false, MONO, R, 1>(a, S, sh.alist + wv * kWave, kWave, gcx, gcy, gcz, ip);
        n_app += W;
        drop_round<W>(sh.alist, na);
      }
    }
    if (overflow) {
      atomicOr(&a.dc->err, 4);  // every lane, same bit
      atomicOr(&a.dc->err_sticky, 4);
      na = 0;
      nd = 0;
    }
    {
      const int a0 = na * wv / T, a1 = na * (wv + 1) / T;
      if (a1 > a0)
        batch_p2c<KAHAN, false, MONO, R, 1>(a, S, sh.alist + a0, a1 - a0, gcx, gcy, gcz, ip);
      const int d0 = nd * wv / T, d1 = nd * (wv + 1) / T;
      if (d1 > d0)
        batch_p2p<KAHAN, false, R, 1>(a, S, sh.dlist + d0, d1 - d0, gcx, gcy, gcz, ip);
      n_app += na;
      n_dir += nd;
    }
    __syncthreads();   // every wave is done with its stage
    // the waves' sums, in the order of the waves
    const Acc4T<R> s = ip.s[0], c = ip.c[0];
    sh.sum[wv][0][lane] = KAHAN ? (double)s.x - (double)c.x : (double)s.x;
    sh.sum[wv][1][lane] = KAHAN ? (double)s.y - (double)c.y : (double)s.y;
    sh.sum[wv][2][lane] = KAHAN ? (double)s.z - (double)c.z : (double)s.z;
    sh.sum[wv][3][lane] = KAHAN ? (double)s.w - (double)c.w : (double)s.w;
    __syncthreads();
    if (wv == 0) {
      double t[4] = {0.0, 0.0, 0.0, 0.0};
      const bool valid = lane < np;
      for (int w = 0; w < T; w++)
        for (int k = 0; k < slices; k++)   // copies of a small group
          for (int q = 0; q < 4; q++) t[q] += sh.sum[w][q][valid ? lane + k * np : lane];
      const Acc4T<R> res = Acc4T<R>{(R)t[0], (R)t[1], (R)t[2], (R)t[3]};
      a.acc[valid ? pbeg + lane : a.n + lane] = make_v4<R>(res.x, res.y, res.z, res.w);
      const double gp = wave_sum(valid ? (double)pi.w * (double)res.w : 0.0);
      a.gcounts[g] = overflow ? make_int2(-1, -1) : make_int2(n_app, n_dir);
      a.gpot[g] = gp;
      atomicMax(&a.dc->stack_max, lane == 0 ? deepest : 0);
      atomicMax(&a.dc->stack_hw, lane == 0 ? deepest : 0);
    }
    __syncthreads();   // the stack and the sums are free for the next group
  }
}

// Interaction statistics (code/computeForces.cu:567-609, :701-715): per valid
// i-particle its group's counts; {direct_sum, direct_max, approx_sum,
// approx_max} and 1/2 sum m phi.  kWalkStatBlocks blocks reduce contiguous
// group ranges, one block combines their partials; up to kStatSmall particles one block
// does it all (2^16: 9 -> 5 us).  A fixed order, so the FP64 potential sum is the same on every
// run.
constexpr int kStatSmall = 1 << 17;
constexpr int kStatThreads = 1024;
struct WStat {
  unsigned long long ds, as;
  unsigned int dm, am;
  double p;
};

// The block's total in thread 0.
__device__ __forceinline__ WStat block_stats(WStat v, WStat *sh) {
  v.ds = wave_sum(v.ds);
  v.as = wave_sum(v.as);
  v.p = wave_sum(v.p);
  for (int m = 32; m >= 1; m >>= 1) {
    v.dm = max(v.dm, (unsigned int)__shfl_xor((int)v.dm, m, kWave));
    v.am = max(v.am, (unsigned int)__shfl_xor((int)v.am, m, kWave));
  }
  const int w = threadIdx.x >> 6;
  if (lane_id() == 0) sh[w] = v;
  __syncthreads();
  if (threadIdx.x == 0) {
    for (int k = 1; k < (int)(blockDim.x >> 6); k++) {
      v.ds += sh[k].ds; v.as += sh[k].as; v.p += sh[k].p;
      v.dm = max(v.dm, sh[k].dm); v.am = max(v.am, sh[k].am);
    }
  }
  return v;
}

// This thread's share of groups [g0, g1).
__device__ __forceinline__ WStat group_stats(const int2 *__restrict__ groups,
                                             const int2 *__restrict__ gcounts,
                                             const double *__restrict__ gpot, int g0, int g1) {
  WStat v = {0ull, 0ull, 0u, 0u, 0.0};
  for (int g = g0 + threadIdx.x; g < g1; g += blockDim.x) {
    const int2 c = gcounts[g];
    const int np = groups[g].y;
    v.ds += (unsigned long long)c.y * (unsigned long long)np;
    v.as += (unsigned long long)c.x * (unsigned long long)np;
    v.dm = max(v.dm, (unsigned int)c.y);
    v.am = max(v.am, (unsigned int)c.x);
    v.p += gpot[g];
  }
  return v;
}

__device__ __forceinline__ void put_stats(DevCounters *dc, const WStat &v) {
  dc->wstats[0] = v.ds; dc->wstats[1] = v.dm; dc->wstats[2] = v.as; dc->wstats[3] = v.am;
  dc->wpot = 0.5 * v.p;
}

__global__ __launch_bounds__(kStatThreads) void k_walk_stats(const int2 *__restrict__ groups,
                                                             const int2 *__restrict__ gcounts,
                                                             const double *__restrict__ gpot,
                                                             DevCounters *dc, const int *run_if,
                                                             DevCounters *host) {
  if (run_if && *run_if == 0) return;   // (host is null then)
  __shared__ WStat sh[kStatThreads / kWave];
  const WStat v = block_stats(group_stats(groups, gcounts, gpot, 0, dc->ngroups), sh);
  if (threadIdx.x == 0) {
    put_stats(dc, v);
    __threadfence();
  }
  __syncthreads();
  write_counters(dc, host);
}

__global__ __launch_bounds__(kBlock) void k_walk_stats_part(const int2 *__restrict__ groups,
                                                           const int2 *__restrict__ gcounts,
                                                           const double *__restrict__ gpot,
                                                           const DevCounters *dc, WStat *part,
                                                           const int *run_if) {
  if (run_if && *run_if == 0) return;
  __shared__ WStat sh[kWavesPerBlock];
  const int ng = dc->ngroups;
  const int chunk = (ng + gridDim.x - 1) / gridDim.x;
  const int g0 = blockIdx.x * chunk, g1 = min(ng, g0 + chunk);
  const WStat v = block_stats(group_stats(groups, gcounts, gpot, g0, g1), sh);
  if (threadIdx.x == 0) part[blockIdx.x] = v;
}

__global__ __launch_bounds__(kBlock) void k_walk_stats_final(const WStat *__restrict__ part,
                                                            DevCounters *dc, const int *run_if) {
  if (run_if && *run_if == 0) return;
  __shared__ WStat sh[kWavesPerBlock];
  WStat v = {0ull, 0ull, 0u, 0u, 0.0};
  for (int k = threadIdx.x; k < kWalkStatBlocks; k += kBlock) {
    const WStat q = part[k];
    v.ds += q.ds; v.as += q.as; v.p += q.p;
    v.dm = max(v.dm, q.dm); v.am = max(v.am, q.am);
  }
  v = block_stats(v, sh);
  if (threadIdx.x == 0) put_stats(dc, v);
}

// clear: the sticky state too, where the walk is the first launch of an API call.
__global__ void k_walk_reset(DevCounters *dc, const int *run_if, bool clear) {
  if (threadIdx.x == 0 && !(run_if && *run_if == 0)) {
    reset_walk(dc);
    if (clear) clear_sticky(dc);
  }
}

}  // namespace

namespace {

template <typename R>
WalkArgs<R> walk_args(Ctx &c, const int *run_if) {
  WalkArgs<R> a;
  a.n = c.n;
  a.nsys = c.nsys;
  a.eps2 = (R)c.eps * (R)c.eps;
  a.groups = c.groups;
  a.group_sys = c.group_sys;
  a.root_cells = c.root_cells;
  a.pos_ph = as4<R>(c.pos_ph);
  a.pos_tree = as4<R>(c.pos);
  a.cells = c.cells;
  a.csize = as4<R>(c.csize);
  a.cmono = as4<R>(c.cmono);
  a.cq0 = as4<R>(c.cq0);
  a.cq1 = as2<R>(c.cq1);
  a.cwalk = as4<R>(c.cwalk);
  a.cls = c.cls;
  a.sys_scale = c.sys_scale;
  a.mlp = c.mlp_dev;
  a.shift = c.learn_shift;
  a.it_min = 1.0f / c.learn_theta_hi;
  a.it_max = 1.0f / c.learn_theta_lo;
  a.acc = as4<R>(c.acc);
  a.gcounts = c.gcounts;
  a.gpot = c.gpot;
  a.stack = c.stack;
  a.stack_ints = c.stack_ints;
  a.lstk_cap = c.lds_stack;
  a.run_if = run_if;
  a.dc = c.dc;
  return a;
}

}  // namespace

// Whether a forest's groups are many and each has little to do.  A team takes its
// barriers and, with the learned angle, four network evaluations for cells that fill
// one; and the wave walk has enough groups to fill the chip.  Fixed angle / learned /
// FP64, teams then waves (us): 256 systems of 1024 1186 1491 / 1768 1510 / 1737 1539, 512
// of 1024 2280 2476 / 3382 2465 / 3330 2498, 32 of 16384 1684 1370 / 1823 1311 / 2758
// 2286, 200 of 1000 927 1272 / 1386 1284 / 1359 1313; 140 of 1000 (-) / 1005 1062 / 984
// 1095, 100 of 2000 654 979 / 923 983 / 1008 1024, 4 of 65536 953 1017 / 841 955 / 1784
// 1693, 128 of 1024 654 1016 / 947 1018 / 922 1049.  At 8 digits a group is a particle or
// two, fixed angle: 512 of 1024 10712 9409, 32 of 16384 6849 4864, but 2048 of 128, whose
// groups are as small at 5 digits, 4645 5566.
static bool many_small_walks(const Ctx &c) {
  if (c.nsys == 1 || c.n <= 1 << 17) return false;
  const bool learned = c.opening == 1 && c.have_mlp;
  if (learned || c.fp64) return c.nsys > 160 || c.n > 1 << 18;
  return c.group_mode == 0 && c.level_split > 6 && c.n / c.nsys >= 512;
}

// Whether the blocks walk groups as teams: below the sizes at which one wave per
// group fills the chip evenly.  Walk times on Plummer spheres (theta 0.5), one wave
// per group / teams: 2^10 509 / 44 us, 2^16 753 / 267, 2^18 1060 / 881, 2^19 1789 /
// 1684, 2^20 3112 / 3398; learned angle 2^18 845 / 613, 2^19 1186 / 1141, 2^20 1910 /
// 2072; FP64 2^18 1816 / 1659, 2^19 3426 / 3150.  (Teams of 2 and 8 waves were
// slower than of 4; with the groups cut into one range per XCD 2^16 took 407 us.)
bool walk_as_team(const Ctx &c) {
  return c.n <= 1 << 19 && !many_small_walks(c) && c.walk_variant == 0 && !c.wave_walk &&
         c.lds_stack == kLdsStack && c.stack_ints >= kSafeStack;
}

namespace {

// variant 0: LDS j-data, one i-particle per lane; 1: scalar-load j-data, one
// i-particle per lane; 2: two i-particles per lane, batches split between the
// half-waves (LDS j-data)
template <bool KAHAN, bool LEARN, bool MONO>
auto wave_kernel(int variant) {
  if constexpr (!MONO) {
    if (variant == 1) return k_walk<float, KAHAN, true, LEARN, MONO, 1>;
  }
  return variant == 2 ? k_walk<float, KAHAN, false, LEARN, MONO, 2>
                      : k_walk<float, KAHAN, false, LEARN, MONO, 1>;
}

template <bool KAHAN, bool LEARN, bool MONO>
auto float_kernel(bool team, int variant) {
  return team ? k_walk_team<float, KAHAN, LEARN, MONO> : wave_kernel<KAHAN, LEARN, MONO>(variant);
}

template <bool KAHAN>
auto float_kernel_of(const Ctx &c, bool team) {
  if (!c.quadrupole) return float_kernel<KAHAN, false, true>(team, c.walk_variant);
  if (c.opening == 1 && c.have_mlp) return float_kernel<KAHAN, true, false>(team, c.walk_variant);
  return float_kernel<KAHAN, false, false>(team, c.walk_variant);
}

template <bool MONO>
auto double_kernel(bool team) {
  return team ? k_walk_team<double, false, false, MONO>
              : k_walk<double, false, false, false, MONO, 1>;
}

}  // namespace

bool walk_stats_in_one(const Ctx &c) { return c.n <= kStatSmall; }

void launch_walk(Ctx &c, const int *run_if, bool clear, bool read, bool reset) {
  c.wstats_valid = false;   // they change with this walk
  const bool team = walk_as_team(c);
  const dim3 blocks(c.walk_blocks), threads(kBlock);
  if (reset)
    hipLaunchKernelGGL(k_walk_reset, dim3(1), dim3(64), 0, c.stream, c.dc, run_if, clear);
  if (c.opening == 1 && !c.fp64) launch_sys_scale(c);   // the learned angle's scales
  if (c.fp64) {
    // Treecode<double>: one i-particle per lane, LDS j-data, FP64 sums
    auto kern = c.quadrupole ? double_kernel<false>(team) : double_kernel<true>(team);
    hipLaunchKernelGGL(kern, blocks, threads, 0, c.stream, walk_args<double>(c, run_if));
  } else {
    auto kern = c.kahan ? float_kernel_of<true>(c, team) : float_kernel_of<false>(c, team);
    hipLaunchKernelGGL(kern, blocks, threads, 0, c.stream, walk_args<float>(c, run_if));
  }
  if (walk_stats_in_one(c)) {
    hipLaunchKernelGGL(k_walk_stats, dim3(1), dim3(kStatThreads), 0, c.stream, c.groups, c.gcounts,
                       c.gpot, c.dc, run_if, read ? c.pinned_dc : nullptr);
    return;
  }
  WStat *part = reinterpret_cast<WStat *>(c.d_wpart);
  hipLaunchKernelGGL(k_walk_stats_part, dim3(kWalkStatBlocks), dim3(kBlock), 0, c.stream, c.groups,
                     c.gcounts, c.gpot, c.dc, part, run_if);
  hipLaunchKernelGGL(k_walk_stats_final, dim3(1), dim3(kBlock), 0, c.stream, part, c.dc, run_if);
}

}  // namespace bt
