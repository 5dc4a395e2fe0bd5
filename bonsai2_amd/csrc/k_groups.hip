// k_groups.hip -- makeGroups on CDNA4 (reference code/makeGroups.cu:236-341).
//
// PH keys of the tree-ordered particles (code/makeGroups.cu:108-135, the
// Hilbert state machine of :19-106), a stable radix sort carrying the tree
// index (:270-277), the gather into PH order (:280), then groups: every run
// of equal keys masked to the top level_split octal digits (:137-192) is cut
// into chunks of ncrit (:196-223).  The reference finds run bounds with two
// inclusive_scan_by_key calls and takes group slots from an atomic counter;
// here each tile of particles finds the start of the run it begins in by a
// search, and a scan of the tiles' group counts gives deterministic group slots
// in PH order.
#include "bt_device.h"
#include "bt_internal.h"

namespace bt {

namespace {

constexpr int kBlock = 256;

// Output digit per Hilbert index (x<<2 | y<<1 | z): {0,1,7,6,3,2,4,5}, packed
// 3 bits per entry.
constexpr uint32_t kHilbertDigits = (0u << 0) | (1u << 3) | (7u << 6) | (6u << 9) | (3u << 12) |
                                    (2u << 15) | (4u << 18) | (5u << 21);

__device__ __forceinline__ uint64_t hilbert_key21(int x, int y, int z) {
  uint64_t key = 0;
#pragma unroll
  for (int lev = 20; lev >= 0; lev--) {
    const int bit = 1 << lev;
    const int idx = ((x & bit) ? 4 : 0) | ((y & bit) ? 2 : 0) | ((z & bit) ? 1 : 0);
    int nx = x, ny = y, nz = z;
    if (idx == 0) {               // swap y and z
      ny = z; nz = y;
    } else if (idx == 1 || idx == 5) {  // swap x and y
      nx = y; ny = x;
    } else if (idx == 4 || idx == 6) {  // complement x and z
      nx = ~x; nz = ~z;
    } else if (idx == 3 || idx == 7) {  // x <- ~y, y <- ~x
      nx = ~y; ny = ~x;
    } else {                      // idx 2: y <- ~z, z <- ~y
      ny = ~z; nz = ~y;
    }
    x = nx; y = ny; z = nz;
    key = (key << 3) + ((kHilbertDigits >> (3 * idx)) & 7u);
  }
  return key;
}

template <typename R>
__global__ __launch_bounds__(kBlock) void k_ph_keys(int n, int nsys, const int *__restrict__ off,
                                                    const V4<R> *__restrict__ box,
                                                    const V4<R> *__restrict__ pos,
                                                    uint64_t *__restrict__ keys,
                                                    int *__restrict__ vals, DevCounters *dc) {
  BT_BUILD_PRIO();
  if (blockIdx.x == 0 && threadIdx.x == 0) atomicAnd(&dc->err, ~kShortPh);
  for (int i = blockIdx.x * kBlock + threadIdx.x; i < n; i += gridDim.x * kBlock) {
    const int r = nsys > 1 ? system_of(i, nsys, off) : 0;
    const V4<R> b = box[r];
    const V4<R> p = pos[i];
    int xc, yc, zc;
    {
#pragma clang fp contract(off)
      // code/makeGroups.cu:123-131, evaluated left to right in real_t
      const R inv = R(0.5) / b.w;
      const R bx = b.x - b.w, by = b.y - b.w, bz = b.z - b.w;
      const R scale = R(2097152);  // 1 << 21
      xc = (int)((p.x - bx) * inv * scale);
      yc = (int)((p.y - by) * inv * scale);
      zc = (int)((p.z - bz) * inv * scale);
    }
    keys[i] = hilbert_key21(xc, yc, zc);
    vals[i] = i;
  }
}

// ---- groups of PH-key runs ------------------------------------------------------
//
// Three launches: the PH gather together with the group counts of every tile, the
// scan of the counts, and the groups.  A particle begins a group iff its distance
// from the start of its run (equal masked keys within a system) is a multiple of
// NCRIT.  Run starts are bits of a tile; the run a tile begins in may have started
// in any tile before it, so a wave looks for it with a 64-way search (4 dependent
// loads at 2^24 keys).  A group ends at the next run start or after NCRIT <= 64
// particles, so a tile needs one word of bits beyond its own.  Bound by the gather.
// (Run starts, a maximum scan, flags, a sum scan, emission and sizes as launches of
// their own took 9 of them, 0.25 ms at 2^24 particles, and 30 us at 2^10.)

constexpr int kGroupTile = 1024;
constexpr int kTileWords = kGroupTile / kWave;
constexpr int kScanThreads = 1024, kScanPer = 4;

struct GroupArgs {
  int n, nsys, ncrit, ntiles, cap;
  const int *off;
  const uint64_t *keys;   // in order as far as the mask goes
  uint64_t mask;
  // a short sort's pairs and where they go (low = 0: keys and perm are final)
  int low;
  const int *perm;
  uint64_t *sorted_keys;
  int *sorted_perm;
  int *count;      // groups of each tile, then their prefixes
  int *carry;      // start of the run each tile begins in
  int2 *groups;
  int *group_sys;
  DevCounters *dc;
  DevCounters *host;   // pinned, or null
};

// Whether particle i starts a run; the ones past the last do.
template <bool FOREST>
__device__ __forceinline__ bool run_start(const GroupArgs &a, int i) {
  if (i == 0 || i >= a.n) return true;
  if ((a.keys[i] & a.mask) != (a.keys[i - 1] & a.mask)) return true;
  return FOREST && system_of(i, a.nsys, a.off) != system_of(i - 1, a.nsys, a.off);
}

// The first particle of particle i's run (all lanes of the wave, same i): the
// masked keys of a system do not decrease.
template <bool FOREST>
__device__ __forceinline__ int find_run_start(const GroupArgs &a, int i) {
  const uint64_t m = a.keys[i] & a.mask;
  int lo = FOREST ? a.off[system_of(i, a.nsys, a.off)] : 0, hi = i;   // in [lo, hi]
  while (lo < hi) {
    const int step = (hi - lo + kWave - 1) / kWave;
    const int p = lo + lane_id() * step;
    const uint64_t in_run = ballot64(p < hi && (a.keys[p] & a.mask) >= m);
    if (in_run == 0) {
      lo = min(hi, lo + ((hi - lo - 1) / step) * step + 1);   // past the last one looked at
    } else {
      const int f = __ffsll((unsigned long long)in_run) - 1;
      hi = lo + f * step;
      lo = f > 0 ? hi - step + 1 : lo;
    }
  }
  return lo;
}

// Bits and run starts of one tile: bits[k] for particles t0 + 64 k.., k <= kTileWords;
// before[k]: the last run start before word k.
struct GroupTile {
  uint64_t bits[kTileWords + 1];
  int before[kTileWords];
  int wave_sum[kBlock / kWave];
};

template <bool FOREST>
__device__ __forceinline__ void load_group_tile(const GroupArgs &a, int t0, int carry,
                                                GroupTile &T) {
  const int lane = lane_id(), w = threadIdx.x >> 6;
  for (int k = w; k <= kTileWords; k += kBlock / kWave) {
    const uint64_t b = ballot64(run_start<FOREST>(a, t0 + k * kWave + lane));
    if (lane == 0) T.bits[k] = b;
  }
  __syncthreads();
  if (w == 0) {
    const uint64_t b = lane < kTileWords ? T.bits[lane] : 0;
    int last = b != 0 ? t0 + lane * kWave + 63 - __clzll((long long)b) : carry;
    // inclusive maximum over the words (a run start is never before an earlier one)
    for (int d = 1; d < kTileWords; d <<= 1) {
      const int v = __shfl_up(last, d, kWave);
      if (lane >= d) last = max(last, v);
    }
    const int v = __shfl_up(last, 1, kWave);
    if (lane < kTileWords) T.before[lane] = lane == 0 ? carry : v;
  }
  __syncthreads();
}

// Whether particle t0 + 64 k + lane begins a group.
__device__ __forceinline__ bool begins_group(const GroupArgs &a, int t0, int k,
                                             const GroupTile &T) {
  const int lane = lane_id(), i = t0 + k * kWave + lane;
  const uint64_t upto = T.bits[k] & (lanemask_lt() | (1ull << lane));
  const int start = upto != 0 ? t0 + k * kWave + 63 - __clzll((long long)upto) : T.before[k];
  return i < a.n && (unsigned)(i - start) % (unsigned)a.ncrit == 0;
}

template <typename T, bool FOREST>
__global__ __launch_bounds__(kBlock) void k_gather_count(GroupArgs a, const T *__restrict__ pos,
                                                         const int *__restrict__ id,
                                                         T *__restrict__ pos_ph,
                                                         int *__restrict__ id_ph) {
  BT_BUILD_PRIO();
  __shared__ GroupTile tile;
  const int t0 = blockIdx.x * kGroupTile;
  const int lane = lane_id(), w = threadIdx.x >> 6;
#pragma unroll
  for (int r = 0; r < kGroupTile / kBlock; r++) {
    const int i = t0 + r * kBlock + threadIdx.x;
    if (i < a.n) {
      const int j = a.perm[i];
      int dst = i;
      if (a.low > 0) {
        const uint64_t key = a.keys[i];
        bool ok = true;
        const int sys = FOREST ? system_of(i, a.nsys, a.off) : 0;
        dst = place_in_run(i, FOREST ? a.off[sys] : 0, FOREST ? a.off[sys + 1] : a.n, a.low, a.keys,
                           key, ok);
        if (!ok) {
          atomicOr(&a.dc->err, kShortPh);
          atomicOr(&a.dc->err_sticky, kShortPh);
          dst = i;   // any order: the walk does nothing
        }
        a.sorted_keys[dst] = key;
        a.sorted_perm[dst] = j;
      }
      pos_ph[dst] = pos[j];
      id_ph[dst] = id[j];
    }
  }
  const int carry = find_run_start<FOREST>(a, t0);
  load_group_tile<FOREST>(a, t0, carry, tile);
  int cnt = 0;
  for (int k = w; k < kTileWords; k += kBlock / kWave)
    cnt += __popcll(ballot64(begins_group(a, t0, k, tile)));
  if (lane == 0) tile.wave_sum[w] = cnt;
  __syncthreads();
  if (threadIdx.x == 0) {
    int s = 0;
    for (int k = 0; k < kBlock / kWave; k++) s += tile.wave_sum[k];
    a.count[blockIdx.x] = s;
    a.carry[blockIdx.x] = carry;
  }
}

// One block: the tiles' counts to prefixes, the number of groups to the counters.
__global__ __launch_bounds__(kScanThreads) void k_group_scan(GroupArgs a) {
  BT_BUILD_PRIO();
  __shared__ int shw[kScanThreads / kWave];
  const int w = threadIdx.x >> 6;
  int carry = 0;
  for (int b0 = 0; b0 < a.ntiles; b0 += kScanThreads * kScanPer) {
    int v[kScanPer], own = 0;
#pragma unroll
    for (int k = 0; k < kScanPer; k++) {
      const int i = b0 + threadIdx.x * kScanPer + k;
      v[k] = i < a.ntiles ? a.count[i] : 0;
      own += v[k];
    }
    const int incl = wave_incl_scan(own);
    if (lane_id() == kWave - 1) shw[w] = incl;
    __syncthreads();
    int pre = carry, tot = 0;
    for (int k = 0; k < kScanThreads / kWave; k++) {
      if (k < w) pre += shw[k];
      tot += shw[k];
    }
    int run = pre + incl - own;
#pragma unroll
    for (int k = 0; k < kScanPer; k++) {
      const int i = b0 + threadIdx.x * kScanPer + k;
      if (i < a.ntiles) a.count[i] = run;
      run += v[k];
    }
    carry += tot;
    __syncthreads();
  }
  if (threadIdx.x == 0) {
    a.dc->ngroups = carry;
    atomicAnd(&a.dc->err, ~2);   // a new set of groups; the level build may run beside this
  }
}

template <bool FOREST>
__global__ __launch_bounds__(kBlock) void k_group_write(GroupArgs a) {
  BT_BUILD_PRIO();
  // (no more groups than particles: nothing below changes them)
  if (blockIdx.x == 0) write_counters(a.dc, a.host);
  __shared__ GroupTile tile;
  const int t0 = blockIdx.x * kGroupTile;
  const int lane = lane_id(), w = threadIdx.x >> 6;
  load_group_tile<FOREST>(a, t0, a.carry[blockIdx.x], tile);
  // wave w takes a quarter of the words in a row
  constexpr int kPer = kTileWords / (kBlock / kWave);
  uint64_t first[kPer];
  int cnt = 0;
#pragma unroll
  for (int q = 0; q < kPer; q++) {
    first[q] = ballot64(begins_group(a, t0, w * kPer + q, tile));
    cnt += __popcll(first[q]);
  }
  if (lane == 0) tile.wave_sum[w] = cnt;
  __syncthreads();
  int slot = a.count[blockIdx.x];
  for (int k = 0; k < w; k++) slot += tile.wave_sum[k];
#pragma unroll
  for (int q = 0; q < kPer; q++) {
    const int k = w * kPer + q;
    if ((first[q] >> lane) & 1) {
      const int i = t0 + k * kWave + lane;
      const int g = slot + __popcll(first[q] & lanemask_lt());
      // run starts after i: the rest of its word, then the next word
      const uint64_t after = lane == kWave - 1 ? tile.bits[k + 1]
                                               : (tile.bits[k] >> (lane + 1)) |
                                                     (tile.bits[k + 1] << (kWave - 1 - lane));
      const int next = after != 0 ? __ffsll((unsigned long long)after) : kWave;
      if (g < a.cap) {
        a.groups[g] = make_int2(i, min(next, a.ncrit));
        a.group_sys[g] = FOREST ? system_of(i, a.nsys, a.off) : 0;
      } else {
        atomicOr(&a.dc->err, 2);
        atomicOr(&a.dc->err_sticky, 2);
      }
    }
    slot += __popcll(first[q]);
  }
}

__global__ __launch_bounds__(kBlock) void k_group_emit(int n, int nsys, const int *__restrict__ off,
                                                       const int *__restrict__ flag,
                                                       const int *__restrict__ slot,
                                                       int cap, int2 *__restrict__ groups,
                                                       int *__restrict__ group_sys,
                                                       DevCounters *dc) {
  BT_BUILD_PRIO();
  for (int i = blockIdx.x * kBlock + threadIdx.x; i < n; i += gridDim.x * kBlock) {
    if (!flag[i]) continue;
    const int g = slot[i];
    if (g >= cap) {
      { atomicOr(&dc->err, 2); atomicOr(&dc->err_sticky, 2); }
      continue;
    }
    groups[g] = make_int2(i, 0);
    group_sys[g] = nsys > 1 ? system_of(i, nsys, off) : 0;
  }
}

// Groups tile [0, n) in order, so a group ends where the next begins.
__global__ __launch_bounds__(kBlock) void k_group_sizes(int n, int cap, int2 *__restrict__ groups,
                                                        DevCounters *dc) {
  BT_BUILD_PRIO();
  const int ng = min(dc->ngroups, cap);
  for (int g = blockIdx.x * kBlock + threadIdx.x; g < ng; g += gridDim.x * kBlock) {
    const int next = g + 1 < ng ? groups[g + 1].x : n;
    groups[g].y = next - groups[g].x;
  }
}

}  // namespace

void launch_ph_keys(Ctx &c) {
  const dim3 g(grid_for(c.n, kBlock, 8192));
  if (c.fp64)
    hipLaunchKernelGGL(k_ph_keys<double>, g, dim3(kBlock), 0, c.stream, c.n, c.nsys, c.d_off,
                       as4<double>(c.box), as4<double>(c.pos), c.ph_keys, c.perm, c.dc);
  else
    hipLaunchKernelGGL(k_ph_keys<float>, g, dim3(kBlock), 0, c.stream, c.n, c.nsys, c.d_off, c.box,
                       c.pos, c.ph_keys, c.perm, c.dc);
}

// A new set of groups starts without the group error bit.
__global__ void k_groups_init(DevCounters *dc) {
  if (threadIdx.x == 0) atomicAnd(&dc->err, ~2);   // the level build may run beside this
}

// Tree groups: flag the first particle of every group cell.  ncrit = 0: the
// leaves (they tile the particles in tree order).  ncrit > 0: the cells of at
// most ncrit particles whose parent holds more (level-1 cells have no parent
// cell), and the leaves of more than ncrit particles; every particle lies in
// exactly one of them.  A group of more than 64 particles (only a leaf capped
// at the deepest level can be one) cannot be one wave's group: err 2.
__global__ __launch_bounds__(kBlock) void k_tree_group_starts(int cap_cells, int ncrit,
                                                              const uint4 *__restrict__ cells,
                                                              int *__restrict__ flag,
                                                              DevCounters *dc) {
  const int nc = min(dc->ncells, cap_cells);
  for (int i = blockIdx.x * kBlock + threadIdx.x; i < nc; i += gridDim.x * kBlock) {
    const uint4 c = cells[i];
    const int np = (int)c.w - (int)c.z;
    bool group;
    if (ncrit == 0) {
      group = cell_leaf(c);
    } else {
      const int level = (int)(c.x >> 27);
      bool parent_splits = true;
      if (level > 1) {
        const uint4 p = cells[c.x & 0x07FFFFFFu];
        parent_splits = (int)p.w - (int)p.z > ncrit;
      }
      group = (cell_leaf(c) || np <= ncrit) && parent_splits;
    }
    if (!group) continue;
    flag[c.z] = 1;
    if (np > kWave) { atomicOr(&dc->err, 2); atomicOr(&dc->err_sticky, 2); }
  }
}

// The group order of leaf groups is the tree order itself.
template <typename T>
__global__ __launch_bounds__(kBlock) void k_identity_order(int n, const T *__restrict__ pos,
                                                           const int *__restrict__ id,
                                                           int *__restrict__ perm,
                                                           T *__restrict__ pos_g,
                                                           int *__restrict__ id_g) {
  for (int i = blockIdx.x * kBlock + threadIdx.x; i < n; i += gridDim.x * kBlock) {
    perm[i] = i;
    pos_g[i] = pos[i];
    id_g[i] = id[i];
  }
}

void launch_leaf_groups(Ctx &c) {
  const int g = grid_for(c.n, kBlock, 8192);
  hipLaunchKernelGGL(k_groups_init, dim3(1), dim3(64), 0, c.stream, c.dc);
  if (c.fp64)
    hipLaunchKernelGGL(k_identity_order<double4>, dim3(g), dim3(kBlock), 0, c.stream, c.n,
                       as4<double>(c.pos), c.id, c.perm, as4<double>(c.pos_ph), c.id_ph);
  else
    hipLaunchKernelGGL(k_identity_order<float4>, dim3(g), dim3(kBlock), 0, c.stream, c.n, c.pos,
                       c.id, c.perm, c.pos_ph, c.id_ph);
  fill_int(c, c.gtmp0, 0, c.n);
  hipLaunchKernelGGL(k_tree_group_starts, dim3(grid_for(c.cap_cells, kBlock, 8192)), dim3(kBlock),
                     0, c.stream, c.cap_cells, c.group_mode == 2 ? c.ncrit : 0, c.cells, c.gtmp0,
                     c.dc);
  scan_exclusive_sum(c, c.gtmp0, c.gtmp1, c.n, &c.dc->ngroups);
  hipLaunchKernelGGL(k_group_emit, dim3(g), dim3(kBlock), 0, c.stream, c.n, c.nsys, c.d_off,
                     c.gtmp0, c.gtmp1, c.cap_groups, c.groups, c.group_sys, c.dc);
  hipLaunchKernelGGL(k_group_sizes, dim3(grid_for(c.cap_groups, kBlock, 4096)), dim3(kBlock), 0,
                     c.stream, c.n, c.cap_groups, c.groups, c.dc);
}

void launch_groups(Ctx &c, bool read) {
  const int ls = c.level_split < 1 ? 1 : c.level_split;
  GroupArgs a;
  a.n = c.n;
  a.nsys = c.nsys;
  a.ncrit = c.ncrit;
  a.ntiles = (c.n + kGroupTile - 1) / kGroupTile;
  a.cap = c.cap_groups;
  a.off = c.d_off;
  a.low = c.ph_low;
  a.keys = a.low > 0 ? c.keyB : c.ph_keys;
  a.perm = a.low > 0 ? c.valB : c.perm;
  a.sorted_keys = c.ph_keys;
  a.sorted_perm = c.perm;
  a.mask = 0;  // top ls octal digits of the 63-bit key (code/makeGroups.cu:259-266)
  for (int i = 0; i < 21; i++) {
    a.mask <<= 3;
    if (i < ls) a.mask |= 7;
  }
  a.count = c.gtmp0;
  a.carry = c.gtmp1;
  a.groups = c.groups;
  a.group_sys = c.group_sys;
  a.dc = c.dc;
  a.host = read ? c.pinned_dc : nullptr;
  const dim3 tiles(a.ntiles);
  const bool forest = c.nsys > 1;
  if (c.fp64) {
    auto kern = forest ? k_gather_count<double4, true> : k_gather_count<double4, false>;
    hipLaunchKernelGGL(kern, tiles, dim3(kBlock), 0, c.stream, a, as4<double>(c.pos), c.id,
                       as4<double>(c.pos_ph), c.id_ph);
  } else {
    auto kern = forest ? k_gather_count<float4, true> : k_gather_count<float4, false>;
    hipLaunchKernelGGL(kern, tiles, dim3(kBlock), 0, c.stream, a, c.pos, c.id, c.pos_ph,
                       c.id_ph);
  }
  hipLaunchKernelGGL(k_group_scan, dim3(1), dim3(kScanThreads), 0, c.stream, a);
  hipLaunchKernelGGL(forest ? k_group_write<true> : k_group_write<false>, tiles, dim3(kBlock), 0,
                     c.stream, a);
}

}  // namespace bt
