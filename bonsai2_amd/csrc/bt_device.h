// bt_device.h -- wave64 helpers shared by the CDNA4 kernels.
#pragma once
#include <hip/hip_runtime.h>
#include <stdint.h>

namespace bt {

constexpr int kWave = 64;
constexpr int kMaxLevel = 21;  // octant digits in a 63-bit geometric key

// The kernels of the build (box, keys, sorts, gathers, levels, multipoles,
// groups) raise their waves' issue priority above the default 0: during a
// step the learned walk's FP64 check sum runs beside them on another stream,
// and on a SIMD they share, the build's latency-bound waves then issue ahead
// of its arithmetic.
#ifndef BT_BUILD_WAVE_PRIO
#define BT_BUILD_WAVE_PRIO 1
#endif
#define BT_BUILD_PRIO() __builtin_amdgcn_s_setprio(BT_BUILD_WAVE_PRIO)

__device__ __forceinline__ int lane_id() { return (int)(threadIdx.x & (kWave - 1)); }

__device__ __forceinline__ uint64_t ballot64(bool p) { return (uint64_t)__ballot(p); }

__device__ __forceinline__ uint64_t lanemask_lt() {
  return (1ull << lane_id()) - 1ull;
}

// Which of the lanes of `peers` have this lane's digit (8 bits), and how many of a
// mask's lanes come before this one.  In this form a bit takes 4 vector instructions
// (the sign-extended bit, its ballot, and one three-input operation for each half of
// the mask), with 64-bit selects it took 9.
__device__ __forceinline__ uint64_t same_digit(uint64_t peers, int d) {
  uint32_t lo = (uint32_t)peers, hi = (uint32_t)(peers >> 32);
#pragma unroll
  for (int b = 0; b < 8; b++) {
    const uint32_t s = (uint32_t)((int)((uint32_t)d << (31 - b)) >> 31);
    const uint64_t m = ballot64(s != 0);
    lo &= ~((uint32_t)m ^ s);
    hi &= ~((uint32_t)(m >> 32) ^ s);
  }
  return (uint64_t)hi << 32 | lo;
}
__device__ __forceinline__ int lanes_before(uint64_t mask) {
  return (int)__builtin_amdgcn_mbcnt_hi((uint32_t)(mask >> 32),
                                        __builtin_amdgcn_mbcnt_lo((uint32_t)mask, 0u));
}

// Orders LDS accesses of different lanes of one wave: all lanes' prior LDS
// writes are visible to all lanes' later LDS reads (a wave executes its LDS
// instructions in order; this stops the compiler from moving them).
__device__ __forceinline__ void wave_lds_sync() {
  __builtin_amdgcn_fence(__ATOMIC_RELEASE, "wavefront");
  __builtin_amdgcn_wave_barrier();
  __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "wavefront");
}

template <typename T>
__device__ __forceinline__ T wave_bcast(T v, int src) { return __shfl(v, src, kWave); }

__device__ __forceinline__ int wave_uniform(int v) { return __builtin_amdgcn_readfirstlane(v); }

template <typename T>
__device__ __forceinline__ T wave_sum(T v) {
#pragma unroll
  for (int m = 32; m >= 1; m >>= 1) v += __shfl_xor(v, m, kWave);
  return v;
}
// One step of a wave-wide scan or reduction: the value CTRL moves to this lane
// (DPP: row_shr:k within rows of 16 lanes, row_bcast:15/31 from the last lane of
// one row or two rows to the next), `old` in lanes that nothing moves to and in
// rows outside ROWS.  One VALU operation, where a shuffle goes through the LDS
// crossbar (about 100 cycles before its result can be used).  All lanes active.
template <int CTRL, int ROWS = 0xF>
__device__ __forceinline__ int dpp_move(int old, int v) {
  return __builtin_amdgcn_update_dpp(old, v, CTRL, ROWS, 0xF, false);
}
template <int CTRL, int ROWS = 0xF>
__device__ __forceinline__ float dpp_move(float old, float v) {
  return __builtin_bit_cast(
      float, dpp_move<CTRL, ROWS>(__builtin_bit_cast(int, old), __builtin_bit_cast(int, v)));
}
template <int CTRL, int ROWS = 0xF>
__device__ __forceinline__ double dpp_move(double old, double v) {
  const long long o = __builtin_bit_cast(long long, old), x = __builtin_bit_cast(long long, v);
  const unsigned lo = (unsigned)dpp_move<CTRL, ROWS>((int)o, (int)x);
  const unsigned hi = (unsigned)dpp_move<CTRL, ROWS>((int)(o >> 32), (int)(x >> 32));
  return __builtin_bit_cast(double, ((unsigned long long)hi << 32) | lo);
}
constexpr int kRowShr = 0x110, kRowBcast15 = 0x142, kRowBcast31 = 0x143;

// Lane 63's value, in every lane.
__device__ __forceinline__ int last_lane(int v) { return __builtin_amdgcn_readlane(v, kWave - 1); }
__device__ __forceinline__ float last_lane(float v) {
  return __builtin_bit_cast(float, last_lane(__builtin_bit_cast(int, v)));
}
__device__ __forceinline__ double last_lane(double v) {
  const long long x = __builtin_bit_cast(long long, v);
  const unsigned lo = (unsigned)last_lane((int)x), hi = (unsigned)last_lane((int)(x >> 32));
  return __builtin_bit_cast(double, ((unsigned long long)hi << 32) | lo);
}

// op over the 64 lanes; op(x, x) = x.
template <typename T, typename Op>
__device__ __forceinline__ T wave_reduce(T v, Op op) {
  v = op(v, dpp_move<kRowShr + 1>(v, v));
  v = op(v, dpp_move<kRowShr + 2>(v, v));
  v = op(v, dpp_move<kRowShr + 4>(v, v));
  v = op(v, dpp_move<kRowShr + 8>(v, v));
  v = op(v, dpp_move<kRowBcast15, 0xA>(v, v));
  v = op(v, dpp_move<kRowBcast31, 0xC>(v, v));
  return last_lane(v);
}

__device__ __forceinline__ int wave_max_int(int v) {
  return wave_reduce(v, [](int a, int b) { return max(a, b); });
}
// Inclusive prefix sum over the 64 lanes.
__device__ __forceinline__ int wave_incl_scan(int v) {
  v += dpp_move<kRowShr + 1>(0, v);
  v += dpp_move<kRowShr + 2>(0, v);
  v += dpp_move<kRowShr + 4>(0, v);
  v += dpp_move<kRowShr + 8>(0, v);
  v += dpp_move<kRowBcast15, 0xA>(0, v);
  v += dpp_move<kRowBcast31, 0xC>(0, v);
  return v;
}

// Vector types of the real type: Treecode<float> (float4 particles and cell
// data) and Treecode<double> (double4).  A context allocates its particle and
// cell arrays with the element size of its real type; kernels view them
// through as4 / as2.
template <typename R> struct RealVec;
template <> struct RealVec<float> { typedef float4 v4; typedef float2 v2; };
template <> struct RealVec<double> { typedef double4 v4; typedef double2 v2; };
template <typename R> using V4 = typename RealVec<R>::v4;
template <typename R> using V2 = typename RealVec<R>::v2;

template <typename R>
__host__ __device__ __forceinline__ V4<R> make_v4(R x, R y, R z, R w) {
  V4<R> v;
  v.x = x; v.y = y; v.z = z; v.w = w;
  return v;
}
template <typename R>
__host__ __device__ __forceinline__ V2<R> make_v2(R x, R y) {
  V2<R> v;
  v.x = x; v.y = y;
  return v;
}
template <typename R, typename P>
__host__ __device__ __forceinline__ V4<R> *as4(P *p) { return reinterpret_cast<V4<R> *>(p); }
template <typename R, typename P>
__host__ __device__ __forceinline__ V2<R> *as2(P *p) { return reinterpret_cast<V2<R> *>(p); }

// min / max of the real type, and over the wave
template <typename R>
__device__ __forceinline__ R rmin(R a, R b) { return fmin(a, b); }
template <typename R>
__device__ __forceinline__ R rmax(R a, R b) { return fmax(a, b); }
template <>
__device__ __forceinline__ float rmin(float a, float b) { return fminf(a, b); }
template <>
__device__ __forceinline__ float rmax(float a, float b) { return fmaxf(a, b); }
template <typename R>
__device__ __forceinline__ R wave_min_r(R v) {
  return wave_reduce(v, [](R a, R b) { return rmin<R>(a, b); });
}
template <typename R>
__device__ __forceinline__ R wave_max_r(R v) {
  return wave_reduce(v, [](R a, R b) { return rmax<R>(a, b); });
}

// System (root) of a particle index: offsets[0..nsys] partition [0, n).  A table behind
// them (system_table) holds the systems of particles 0, 256, 512, ..., so that a search
// runs over those of one such stretch only, mostly a single one.  (Over all 256 systems
// of an ensemble of 4*10^6 it was 8 loads that depend on each other: PH keys 88 -> 62 us,
// a pass's histogram by system 33 -> 15, its scatter 62 -> 35, the groups' gather 122 -> 79.)
constexpr int kSystemStep = 256;
__device__ __forceinline__ int system_of(int i, int nsys, const int *__restrict__ off) {
  const int *stretch = off + nsys + 1 + (unsigned)i / kSystemStep;
  int lo = stretch[0], hi = stretch[1];
  while (lo < hi) {
    const int mid = (lo + hi + 1) >> 1;
    if (off[mid] <= i) lo = mid; else hi = mid - 1;
  }
  return lo;
}

// The place of pair i among pairs sorted by all but the low `low` bits of their keys
// (stably, and within systems, of which this one's pairs are [lo, hi)): pairs that agree
// in the sorted bits form short runs, in which a pair's place is the number of smaller
// keys, ties in their order.  A run of more than kRunMax pairs is not looked through: `ok`
// is cleared, in all of its pairs.  256: an evolving halo and disk of 2^24, whose box
// grows with the particles that leave it, had a run of more than 64 in its 24th step, and
// 8 digits instead of 5 from then on (sorts 1.53 -> 2.47 ms a step); looking through
// longer runs costs its gathers 0.09 ms.  Most pairs have no neighbour in their run: the
// nearest two are read together (2*10^7 ordinary particles: the tree's gather 364 -> 367 us,
// the groups' 400 -> 390), up to kSingly on either side one by one, and those past them
// eight at a time, as the reads' latency is what a long run costs (2^22 particles in clumps
// of 120: build 1.11 -> 0.92 ms, groups 0.93 -> 0.72; 2^20 in clumps of 250 0.50 -> 0.41 and
// 0.57 -> 0.37).
constexpr int kRunMax = 256;
__device__ __forceinline__ int place_in_run(int i, int lo, int hi, int low,
                                            const uint64_t *__restrict__ keys, uint64_t key,
                                            bool &ok) {
  constexpr int kSingly = 8, kAhead = 8;
  auto in_run = [&](uint64_t x) { return ((x ^ key) >> low) == 0; };
  // the nearest two together; most pairs are done with that
  const uint64_t prev = keys[max(i - 1, lo)], next = keys[min(i + 1, hi - 1)];
  int before = i > lo && in_run(prev) ? 1 : 0, after = i + 1 < hi && in_run(next) ? 1 : 0;
  int place = i;
  if (before + after == 0) return place;
  place += (after && next < key ? 1 : 0) - (before && prev > key ? 1 : 0);
  if (before) {
    for (int k = i - 2; k >= lo; k--) {
      const uint64_t x = keys[k];
      if (!in_run(x)) break;
      place -= x > key ? 1 : 0;
      if (++before >= kSingly) break;
    }
  }
  if (after) {
    for (int k = i + 2; k < hi; k++) {
      const uint64_t x = keys[k];
      if (!in_run(x)) break;
      place += x < key ? 1 : 0;
      if (++after >= kSingly) break;
    }
  }
  if (max(before, after) < kSingly) return place;
  if (before >= kSingly) {
    bool in = true;
    for (int k = i - 1 - kSingly; in && before < kRunMax; k -= kAhead) {
      uint64_t x[kAhead];
#pragma unroll
      for (int q = 0; q < kAhead; q++) x[q] = keys[max(k - q, lo)];
#pragma unroll
      for (int q = 0; q < kAhead; q++) {
        in = in && k - q >= lo && in_run(x[q]);
        place -= in && x[q] > key ? 1 : 0;
        before += in ? 1 : 0;
      }
    }
  }
  if (after >= kSingly) {
    bool in = true;
    for (int k = i + 1 + kSingly; in && before + after < kRunMax; k += kAhead) {
      uint64_t x[kAhead];
#pragma unroll
      for (int q = 0; q < kAhead; q++) x[q] = keys[min(k + q, hi - 1)];
#pragma unroll
      for (int q = 0; q < kAhead; q++) {
        in = in && k + q < hi && in_run(x[q]);
        place += in && x[q] < key ? 1 : 0;
        after += in ? 1 : 0;
      }
    }
  }
  if (before + after >= kRunMax) ok = false;
  return place;
}

// CellData bit layout (reference code/Treecode.h:45-89):
//   x = parent | level << 27; y = first | (nchild-1) << 29, or 0xFFFFFFFF for
//   a leaf; z = pbeg; w = pend (half-open, tree order).
__device__ __forceinline__ bool cell_leaf(const uint4 &c) { return c.y == 0xFFFFFFFFu; }
__device__ __forceinline__ int cell_first(const uint4 &c) { return (int)(c.y & 0x1FFFFFFFu); }
__device__ __forceinline__ int cell_nchild(const uint4 &c) { return (int)(c.y >> 29) + 1; }
__device__ __forceinline__ uint32_t cell_pack_y(int first, int nchild) {
  return (uint32_t)first | ((uint32_t)(nchild - 1) << 29);
}

}  // namespace bt
