// k_tree.hip -- buildTree and computeMultipoles on CDNA4.
//
// The reference builds the octree by recursive dynamic parallelism
// (code/buildTree.cu:170-584: every split cell's last block launches the
// children's grid from the device).  HIP has no device-side launch, so the
// build here is key-based:
//
//   1. root box per system (code/buildTree.cu:80-166), bit-exact float ops;
//   2. per particle, its geometric key: the 21 octant digits it takes down the
//      same float ChildBox/Octant recursion the reference evaluates per cell
//      (code/Particle4.h:129-148, code/buildTree.cu:233-247);
//   3. a stable radix sort of the keys = the reference's scatter into child
//      ranges in octant order (:444-471), within-leaf order canonical;
//   4. cells: the children of a level-(L-1) cell are the runs of equal digit L
//      inside its particle range; count > NLEAF -> node, 0 < count <= NLEAF ->
//      leaf (:394-395); children of one parent are [nodes in octant order]
//      [leaves in octant order] (:393-400, :549) and levels are contiguous,
//      parents in order (the level sort, :932-951).  All levels are found at
//      once from the sorted keys, in launches whose sizes the host knows, so
//      the whole build can be graph-captured.
//
// Multipoles (code/computeMultipoles.cu:81-190) are computed bottom-up: the
// leaves sum their particles, then the nodes, from the deepest level, combine
// their children with the parallel-axis theorem.  Moments are carried
// relative to a reference point inside the cell's particle bbox (a leaf's
// first particle; a node's first child's reference), so every offset is at
// most the particle extent l and the FP32 sums keep their digits for small
// cells far from the origin and for sparse cells; levels <= kFp64Levels
// combine in FP64.  Outputs keep the reference layout (:180-188).
#include <algorithm>

#include "bt_device.h"
#include "bt_internal.h"

namespace bt {

namespace {

constexpr int kBlock = 256;

// ---- root box -----------------------------------------------------------

template <typename R>
struct Ext {
  R nx, ny, nz, xx, xy, xz;   // min and max per axis
};

template <typename R>
__device__ __forceinline__ void ext_add(Ext<R> &e, R x, R y, R z) {
  e.nx = rmin(e.nx, x); e.ny = rmin(e.ny, y); e.nz = rmin(e.nz, z);
  e.xx = rmax(e.xx, x); e.xy = rmax(e.xy, y); e.xz = rmax(e.xz, z);
}
template <typename R>
__device__ __forceinline__ Ext<R> ext_empty() {
  return Ext<R>{R(1e10), R(1e10), R(1e10), R(-1e10), R(-1e10), R(-1e10)};
}
// Union of two extents, either of which may be empty (min > max): minima with
// minima, maxima with maxima.
template <typename R>
__device__ __forceinline__ void ext_merge(Ext<R> &e, R nx, R ny, R nz, R xx, R xy, R xz) {
  e.nx = rmin(e.nx, nx); e.ny = rmin(e.ny, ny); e.nz = rmin(e.nz, nz);
  e.xx = rmax(e.xx, xx); e.xy = rmax(e.xy, xy); e.xz = rmax(e.xz, xz);
}

// block-wide min/max; the block's result in thread 0
template <typename R>
__device__ __forceinline__ void block_minmax(Ext<R> &e, Ext<R> *sh) {
  e.nx = wave_min_r(e.nx); e.ny = wave_min_r(e.ny); e.nz = wave_min_r(e.nz);
  e.xx = wave_max_r(e.xx); e.xy = wave_max_r(e.xy); e.xz = wave_max_r(e.xz);
  const int w = threadIdx.x >> 6;
  if (lane_id() == 0) sh[w] = e;
  __syncthreads();
  if (threadIdx.x == 0) {
    for (int k = 1; k < (int)(blockDim.x >> 6); k++)
      ext_merge(e, sh[k].nx, sh[k].ny, sh[k].nz, sh[k].xx, sh[k].xy, sh[k].xz);
  }
}

template <typename R>
__global__ __launch_bounds__(kBlock) void k_bbox_partial(const V4<R> *__restrict__ pos,
                                                         const int *__restrict__ off, int nb,
                                                         V4<R> *__restrict__ part) {
  BT_BUILD_PRIO();
  __shared__ Ext<R> sh[kBlock / kWave];
  const int r = blockIdx.y;
  const int b = off[r], e = off[r + 1];
  Ext<R> x = ext_empty<R>();
  for (int i = b + blockIdx.x * kBlock + threadIdx.x; i < e; i += nb * kBlock) {
    const V4<R> p = pos[i];
    ext_add(x, p.x, p.y, p.z);
  }
  block_minmax(x, sh);
  if (threadIdx.x == 0) {
    part[2 * (r * nb + blockIdx.x)] = make_v4<R>(x.nx, x.ny, x.nz, R(0));
    part[2 * (r * nb + blockIdx.x) + 1] = make_v4<R>(x.xx, x.xy, x.xz, R(0));
  }
}

// Box rules of code/buildTree.cu:145-161, same operations in real_t.  (The
// reference's double instantiation would round the extremes to float in its
// float2 block reduction, code/buildTree.cu:102-105; they stay double here.)
template <typename R>
__device__ V4<R> box_from_extent(const Ext<R> &e) {
#pragma clang fp contract(off)
  const R cx = (e.xx + e.nx) * R(0.5), cy = (e.xy + e.ny) * R(0.5), cz = (e.xz + e.nz) * R(0.5);
  const R hx = (e.xx - e.nx) * R(0.5), hy = (e.xy - e.ny) * R(0.5), hz = (e.xz - e.nz) * R(0.5);
  const R h = rmax(hz, rmax(hy, hx));
  R hs = R(1);
  if (h > R(0)) {
    while (hs > h) hs *= R(0.5);
    while (hs < h) hs *= R(2);
  }
  const R hq = hs / R(1048576);
  const long long qx = (long long)(cx / hq), qy = (long long)(cy / hq), qz = (long long)(cz / hq);
  return make_v4<R>(hq * (R)qx, hq * (R)qy, hq * (R)qz, hs);
}

template <typename R>
__global__ __launch_bounds__(kBlock) void k_bbox_final(const V4<R> *__restrict__ part, int nb,
                                                       V4<R> *__restrict__ box) {
  BT_BUILD_PRIO();   // beside the check's sums it took 88 us without, 4 with
  __shared__ Ext<R> sh[kBlock / kWave];
  const int r = blockIdx.x;
  Ext<R> x = ext_empty<R>();
  for (int k = threadIdx.x; k < nb; k += kBlock) {
    const V4<R> a = part[2 * (r * nb + k)], b = part[2 * (r * nb + k) + 1];
    ext_merge(x, a.x, a.y, a.z, b.x, b.y, b.z);   // a block may have had no particles
  }
  block_minmax(x, sh);
  if (threadIdx.x == 0) box[r] = box_from_extent(x);
}

// ---- geometric keys -----------------------------------------------------

// One ChildBox step (code/Particle4.h:138-148): the centre moves by hsize/2.
template <typename R>
__device__ __forceinline__ void child_step(R &cx, R &cy, R &cz, R &h, int o) {
#pragma clang fp contract(off)
  const R s = R(0.5) * h;
  cx = (o & 1) ? cx + s : cx - s;
  cy = (o & 2) ? cy + s : cy - s;
  cz = (o & 4) ? cz + s : cz - s;
  h = s;
}

// BOX: one system whose partial boxes are kBoxParts at most: every wave makes the box of
// them (2^16 particles: 3 + 4 -> 4 us, and a launch gap less).
constexpr int kBoxParts = kWave;
template <typename R, bool BOX>
__global__ __launch_bounds__(kBlock) void k_geo_keys(int n, int nsys, const int *__restrict__ off,
                                                     V4<R> *__restrict__ box,
                                                     const V4<R> *__restrict__ part, int nb,
                                                     const V4<R> *__restrict__ pos,
                                                     uint64_t *__restrict__ keys,
                                                     int *__restrict__ vals, DevCounters *dc) {
  BT_BUILD_PRIO();
  if (blockIdx.x == 0 && threadIdx.x == 0) atomicAnd(&dc->err, ~kShortTree);
  V4<R> own;
  if constexpr (BOX) {
    const int k = min(lane_id(), nb - 1);
    const V4<R> mn = part[2 * k], mx = part[2 * k + 1];
    const Ext<R> e{wave_min_r(mn.x), wave_min_r(mn.y), wave_min_r(mn.z),
                   wave_max_r(mx.x), wave_max_r(mx.y), wave_max_r(mx.z)};
    own = box_from_extent(e);
    if (blockIdx.x == 0 && threadIdx.x == 0) box[0] = own;
  }
  for (int i = blockIdx.x * kBlock + threadIdx.x; i < n; i += gridDim.x * kBlock) {
    const int r = nsys > 1 ? system_of(i, nsys, off) : 0;
    const V4<R> b = BOX ? own : box[r];
    const V4<R> p = pos[i];
    R cx = b.x, cy = b.y, cz = b.z, h = b.w;
    uint64_t k = 0;
#pragma unroll
    for (int l = 0; l < kMaxLevel; l++) {
      // Octant (code/Particle4.h:129-136): bit set iff centre <= pos
      const int o = (int)(cx <= p.x) | ((int)(cy <= p.y) << 1) | ((int)(cz <= p.z) << 2);
      k = (k << 3) | (uint64_t)o;
      child_step(cx, cy, cz, h, o);
    }
    keys[i] = k;
    vals[i] = i;
  }
}

// The particles in the order of their sorted keys.  low > 0: the pairs come from a
// short sort (keys, perm), and their runs are put in order here; sorted_keys receives
// the keys.  IDENT: the ids are the particles' places still, so none is read.  Bound
// by the lines that the permuted reads touch (on a first build, of unordered
// particles, one per 16 B).
template <typename T, bool SHORT, bool FOREST, bool IDENT>
__global__ __launch_bounds__(kBlock) void k_gather3(int n, const int *__restrict__ perm,
                                                    const T *__restrict__ a,
                                                    const T *__restrict__ b,
                                                    const int *__restrict__ c,
                                                    T *__restrict__ a2,
                                                    T *__restrict__ b2,
                                                    int *__restrict__ c2, int low,
                                                    const uint64_t *__restrict__ keys,
                                                    uint64_t *__restrict__ sorted_keys, int nsys,
                                                    const int *__restrict__ off, DevCounters *dc) {
  BT_BUILD_PRIO();
  for (int i = blockIdx.x * kBlock + threadIdx.x; i < n; i += gridDim.x * kBlock) {
    const int j = perm[i];
    int dst = i;
    if (SHORT) {
      const uint64_t key = keys[i];
      bool ok = true;
      const int sys = FOREST ? system_of(i, nsys, off) : 0;
      dst = place_in_run(i, FOREST ? off[sys] : 0, FOREST ? off[sys + 1] : n, low, keys, key, ok);
      if (!ok) {
        atomicOr(&dc->err, kShortTree);
        atomicOr(&dc->err_sticky, kShortTree);
        dst = i;   // any order: what follows does nothing
      }
      sorted_keys[dst] = key;
    }
    a2[dst] = a[j];
    b2[dst] = b[j];
    c2[dst] = IDENT ? j : c[j];
  }
}

// ---- cell emission: every level from the sorted keys at once ---------------
//
// Which cells exist, and where they begin and end, follows from each particle's
// neighbours in key order alone, so no level has to wait for the one above it:
//   * c(i): the octant digits particle i shares with particle i - 1 (0 at a
//     system's first particle);
//   * D(i): the deepest node that holds particle i.  A cell holds more than
//     NLEAF particles iff some window of NLEAF + 1 consecutive particles lies in
//     it, so D(i) is the maximum of the shared digits of keys[k], keys[k + NLEAF]
//     over the windows k in [i - NLEAF, i], at most kMaxLevel - 1 (a level-21
//     cell does not split) and at least 0 (the root always splits,
//     code/buildTree.cu:702).
// Particle i begins the cells of levels c(i) + 1 .. D(i) + 1, the last of them a
// leaf, and ends those of levels c(i) + 1 .. D(i - 1) + 1.  A cell's place in its
// level is the number of beginnings of that level before it, which is the parent
// order with the children of a parent in octant order; only [nodes][leaves]
// within one parent (code/buildTree.cu:393-400, :549) has to be put right after.
// Five launches for any tree: count the beginnings per tile and level, scan them
// over the tiles, write the cells in octant order ("raw" slots), order each
// parent's children, write the cells.  Bound by latency below 2^20 particles and
// by the traffic on keys (8 B per particle, twice) and cells above.
// A launch triple per level with binary searches for the children (64 launches)
// took 0.26 ms at 2^16 and 0.83 ms at 2^24 particles.

// Particles per block: ROUNDS rounds of 64 in a row per wave.  Four are worth the
// window's halo (2 NLEAF keys) and the fewer counts; up to kCellSmall particles, where a
// round's latency is what a tile costs, one
// (count and emit: 7 + 14 -> 4.5 + 7 us at 2^10, 9 + 15 -> 5 + 7.5 at 2^16).
constexpr int kCellRounds = 4;
constexpr int kCellSmall = 1 << 17;
constexpr int kCellRows = kCellCntRows;                // row 0: leaves; row L: cells of level L
static_assert(kCellRows == kMaxLevel + 1, "a row per level and one for the leaves");
constexpr int kMaxLeaf = 64;
constexpr int kScanBlock = 1024, kScanPer = 4;       // the scan of one row over the tiles

struct LevelArgs {
  int nsys, nleaf, cap_cells, n, ntiles;
  const int *off;
  const uint64_t *keys;
  uint4 *cells;
  uint4 *raw;        // octant-order slots: (raw parent | L << 27, first raw child or ~0, begin, end)
  int *fin;          // final slot of each raw slot
  int *nch;          // children of each raw node
  int *arrived;      // per node, for the multipoles: 0
  int *cnt;          // kCellRows x ntiles: counts, then their prefixes over the tiles
  int2 *root_cells;
  int2 *level_beg;
  DevCounters *dc;
  DevCounters *host;   // pinned, or null
};

// Octant digits two 63-bit keys share.
__device__ __forceinline__ int shared_digits(uint64_t a, uint64_t b) {
  const uint64_t x = a ^ b;
  return x == 0 ? kMaxLevel : (__clzll((long long)x) - 1) / 3;
}

// One tile's keys and depths.  Entry j of a window array belongs to particle
// t0 - 1 - NLEAF + j, entry j of depth to particle t0 - 1 + j.
template <int ROUNDS>
struct CellTile {
  static constexpr int kCellTile = ROUNDS * kBlock;
  uint64_t key[kCellTile + 2 * kMaxLeaf + 2];
  int sys[kCellTile + 2 * kMaxLeaf + 2];   // forest: the particle's system
  unsigned char win[2][kCellTile + kMaxLeaf + 2];
  unsigned char depth[kCellTile + 2];
};

// Fills the tile and returns whether one of its windows shares all digits (a
// level-21 cell of more than NLEAF particles).
template <bool FOREST, int ROUNDS>
__device__ __forceinline__ bool load_cell_tile(const LevelArgs &a, int t0, CellTile<ROUNDS> &T) {
  constexpr int kCellTile = ROUNDS * kBlock;
  const int nl = a.nleaf;
  const int k0 = t0 - 1 - nl;   // particle of entry 0
  for (int j = threadIdx.x; j < kCellTile + 2 * nl + 1; j += kBlock) {
    const int i = min(max(k0 + j, 0), a.n - 1);
    T.key[j] = a.keys[i];
    if (FOREST) T.sys[j] = system_of(i, a.nsys, a.off);
  }
  __syncthreads();
  bool full = false;
  const int nw = kCellTile + nl + 1;
  for (int j = threadIdx.x; j < nw; j += kBlock) {
    const int k = k0 + j;
    int w = 0;
    if (k >= 0 && k + nl < a.n && (!FOREST || T.sys[j] == T.sys[j + nl])) {
      w = shared_digits(T.key[j], T.key[j + nl]);
      full |= w == kMaxLevel;
      w = min(w, kMaxLevel - 1);
    }
    T.win[0][j] = (unsigned char)w;
  }
  __syncthreads();
  // maxima over 2, 4, ... consecutive windows; the last power of two within
  // NLEAF + 1 covers them as two overlapping runs
  int cur = 0, len = 1;
  for (; 2 * len <= nl + 1; len *= 2) {
    for (int j = threadIdx.x; j < nw; j += kBlock)
      T.win[cur ^ 1][j] = max(T.win[cur][j], j + len < nw ? T.win[cur][j + len] : (unsigned char)0);
    cur ^= 1;
    __syncthreads();
  }
  for (int j = threadIdx.x; j < kCellTile + 1; j += kBlock)
    T.depth[j] = max(T.win[cur][j], T.win[cur][j + nl + 1 - len]);
  __syncthreads();
  return full;
}

// c(i) and D(i) of particle i = t0 + j; an index past the last particle begins
// nothing (c = kMaxLevel) except that i = n ends what the last particle is in.
template <bool FOREST, int ROUNDS>
__device__ __forceinline__ void cell_span(const LevelArgs &a, const CellTile<ROUNDS> &T, int t0, int j,
                                          int &c, int &d, int &dprev) {
  const int i = t0 + j, e = j + a.nleaf + 1;   // e: entry of particle i in the key array
  d = i < a.n ? (int)T.depth[j + 1] : -1;
  dprev = i > 0 && i <= a.n ? (int)T.depth[j] : -1;
  if (i >= a.n) c = i == a.n ? 0 : kMaxLevel;
  else if (i == 0 || (FOREST && T.sys[e] != T.sys[e - 1])) c = 0;
  else c = shared_digits(T.key[e], T.key[e - 1]);
}

// Lane L of the result counts the beginnings of level L among the wave's
// ROUNDS * 64 particles, lane 0 its leaves.
template <bool FOREST, int ROUNDS>
__device__ __forceinline__ int wave_cell_counts(const LevelArgs &a, const CellTile<ROUNDS> &T,
                                                int t0) {
  const int lane = lane_id(), w = threadIdx.x >> 6;
  int cnt = 0;
#pragma unroll
  for (int r = 0; r < ROUNDS; r++) {
    int c, d, dp;
    cell_span<FOREST, ROUNDS>(a, T, t0, (w * ROUNDS + r) * kWave + lane, c, d, dp);
    const int nleaves = __popcll(ballot64(c <= d));   // d >= 0 for every particle
    cnt += lane == 0 ? nleaves : 0;
    const int hi = wave_max_int(d + 1);
    for (int L = 1; L <= hi; L++) {
      const int m = __popcll(ballot64(c < L && L <= d + 1));
      cnt += lane == L ? m : 0;
    }
  }
  return cnt;
}

template <bool FOREST, int ROUNDS>
__global__ __launch_bounds__(kBlock) void k_cells_count(LevelArgs a) {
  BT_BUILD_PRIO();
  __shared__ CellTile<ROUNDS> T;
  __shared__ int sh[kBlock / kWave][kWave];
  const int t0 = blockIdx.x * (ROUNDS * kBlock);
  if (a.dc->err & kShortTree) {   // keys not in order (set before this launch): no cells
    if (threadIdx.x < kCellRows) a.cnt[threadIdx.x * a.ntiles + blockIdx.x] = 0;
    return;
  }
  load_cell_tile<FOREST, ROUNDS>(a, t0, T);
  sh[threadIdx.x >> 6][lane_id()] = wave_cell_counts<FOREST, ROUNDS>(a, T, t0);
  __syncthreads();
  if (threadIdx.x < kCellRows) {
    int s = 0;
    for (int w = 0; w < kBlock / kWave; w++) s += sh[w][threadIdx.x];
    a.cnt[threadIdx.x * a.ntiles + blockIdx.x] = s;
  }
}

// Block b: exclusive prefix of row b over the tiles, its total in lvl_total[b].
__global__ __launch_bounds__(kScanBlock) void k_cells_scan(LevelArgs a) {
  BT_BUILD_PRIO();
  __shared__ int shw[kScanBlock / kWave];
  int *row = a.cnt + (size_t)blockIdx.x * a.ntiles;
  const int w = threadIdx.x >> 6;
  int carry = 0;
  for (int b0 = 0; b0 < a.ntiles; b0 += kScanBlock * kScanPer) {
    int v[kScanPer], own = 0;
#pragma unroll
    for (int k = 0; k < kScanPer; k++) {
      const int i = b0 + threadIdx.x * kScanPer + k;
      v[k] = i < a.ntiles ? row[i] : 0;
      own += v[k];
    }
    const int incl = wave_incl_scan(own);
    if (lane_id() == kWave - 1) shw[w] = incl;
    __syncthreads();
    int pre = carry, tot = 0;
    for (int k = 0; k < kScanBlock / kWave; k++) {
      if (k < w) pre += shw[k];
      tot += shw[k];
    }
    int run = pre + incl - own;
#pragma unroll
    for (int k = 0; k < kScanPer; k++) {
      const int i = b0 + threadIdx.x * kScanPer + k;
      if (i < a.ntiles) row[i] = run;
      run += v[k];
    }
    carry += tot;
    __syncthreads();
  }
  if (threadIdx.x == 0) {
    a.dc->lvl_total[blockIdx.x] = carry;
    if (blockIdx.x == 0) {
      a.dc->flags = 0;
      atomicAnd(&a.dc->err, ~1);   // other bits belong to phases that may run beside this one
    }
  }
}

// The cells in octant order.  Level L of the loop: a particle that begins a cell
// of level L takes the next slot of the level; it writes the cell one level up
// that begins with it as soon as this one's slot, its first child, is known.
template <bool FOREST, int ROUNDS>
__global__ __launch_bounds__(kBlock) void k_cells_emit(LevelArgs a) {
  BT_BUILD_PRIO();
  __shared__ CellTile<ROUNDS> T;
  __shared__ int sh[kBlock / kWave][kWave];
  DevCounters *dc = a.dc;
  const int t0 = blockIdx.x * (ROUNDS * kBlock);
  const int lane = lane_id(), w = threadIdx.x >> 6;
  const bool sorted = !(dc->err & kShortTree);
  bool full = false;
  if (sorted) {
    full = load_cell_tile<FOREST, ROUNDS>(a, t0, T);
    sh[w][lane] = wave_cell_counts<FOREST, ROUNDS>(a, T, t0);
  }
  // lane L: first slot of level L
  const int tot = lane >= 1 && lane <= kMaxLevel ? dc->lvl_total[lane] : 0;
  const int start = wave_incl_scan(tot) - tot;
  const int total = last_lane(start);
  const bool fits = total <= a.cap_cells;
  if (blockIdx.x == 0 && w == 0) {
    const int nleaves = dc->lvl_total[0];
    const uint64_t filled = ballot64(tot > 0);
    if (lane < kLevels) {
      dc->lvl_start[lane] = fits ? start : 0;
      dc->lvl_count[lane] = fits ? tot : 0;
      a.level_beg[lane] = fits && tot > 0 ? make_int2(start, start + tot - 1) : make_int2(0, 0);
    }
    if (lane == 0) {
      dc->nlevels = fits ? kWave - 1 - __clzll((long long)filled) : 0;
      dc->ncells = fits ? total : 0;
      dc->nnodes = fits ? total - nleaves : 0;
      dc->nleaves = fits ? nleaves : 0;
      if (!fits) {
        atomicOr(&dc->err, 1);
        atomicOr(&dc->err_sticky, 1);
      }
    }
  }
  if (full) atomicOr(&dc->flags, (int)BT_FLAG_DEPTH_CAP);
  if (!fits || !sorted) return;
  __syncthreads();
  // lane L: the next slot of level L for this wave
  int next = lane >= 1 && lane <= kMaxLevel ? start + a.cnt[lane * a.ntiles + blockIdx.x] : 0;
  for (int k = 0; k < w; k++) next += lane >= 1 ? sh[k][lane] : 0;
  for (int r = 0; r < ROUNDS; r++) {
    const int j = (w * ROUNDS + r) * kWave + lane;
    const int i = t0 + j;
    int c, d, dp;
    cell_span<FOREST, ROUNDS>(a, T, t0, j, c, d, dp);
    const int hi = wave_max_int(max(d, dp) + 1);
    uint32_t up = 0;       // raw slot of the cell of level L - 1 that holds this particle
    int mine = -1;         // raw slot of the node of level L - 1 that begins here
    uint32_t mine_x = 0;
    for (int L = 1; L <= hi; L++) {
      const bool begins = c < L && L <= d + 1;
      const uint64_t m = ballot64(begins);
      const int base = __builtin_amdgcn_readlane(next, L);
      const int slot = base + __popcll(m & lanemask_lt());
      if (c < L && L <= dp + 1) a.raw[slot - 1].w = (uint32_t)i;   // ends here
      if (begins) {
        uint3 *rec;
        if (mine >= 0) {
          rec = reinterpret_cast<uint3 *>(a.raw + mine);
          *rec = make_uint3(mine_x, (uint32_t)slot, (uint32_t)i);
        }
        const uint32_t x = up | ((uint32_t)L << 27);
        if (L == d + 1) {
          rec = reinterpret_cast<uint3 *>(a.raw + slot);
          *rec = make_uint3(x, 0xFFFFFFFFu, (uint32_t)i);
        } else {
          mine = slot;
          mine_x = x;
        }
        const int e = j + a.nleaf + 1;   // this particle in the tile's arrays
        if (L == 1 && (i == 0 || (FOREST && T.sys[e] != T.sys[e - 1])))
          a.root_cells[FOREST ? T.sys[e] : 0] = make_int2(slot, 0);
      }
      up = (uint32_t)(begins ? slot : slot - 1);
      next += lane == L ? __popcll(m) : 0;
    }
  }
}

// Children k < nc of one parent from raw slot f on (their last ends at `end`):
// bit k of `nodes` is set if child k is a node.
__device__ __forceinline__ int scan_children(const LevelArgs &a, int f, uint32_t end,
                                             uint32_t &nodes) {
  int nc = 0;
  nodes = 0;
  for (; nc < 8; nc++) {
    const uint4 r = a.raw[f + nc];
    nodes |= (r.y != 0xFFFFFFFFu ? 1u : 0u) << nc;
    if (r.w == end) return nc + 1;
  }
  return nc;
}

__device__ __forceinline__ void place_children(const LevelArgs &a, int f, int nc, uint32_t nodes) {
  const int nn = __popc(nodes);
  for (int k = 0; k < nc; k++) {
    const int before = __popc(nodes & ((1u << k) - 1u));
    a.fin[f + k] = f + ((nodes >> k) & 1u ? before : nn + k - before);
  }
}

// Final slot of every cell: each parent puts its children, which fill a run of
// slots, into the order [nodes][leaves].
__global__ __launch_bounds__(kBlock) void k_cells_place(LevelArgs a) {
  BT_BUILD_PRIO();
  const int nc_all = a.dc->ncells;
  const bool failed = a.dc->err & (1 | kShortTree);
  const int stride = gridDim.x * kBlock;
  for (int s = blockIdx.x * kBlock + threadIdx.x; s < nc_all; s += stride) {
    const uint4 r = a.raw[s];
    if (r.y == 0xFFFFFFFFu) continue;
    uint32_t nodes;
    const int nc = scan_children(a, (int)r.y, r.w, nodes);
    place_children(a, (int)r.y, nc, nodes);
    a.nch[s] = nc;
  }
  for (int r = blockIdx.x * kBlock + threadIdx.x; r < a.nsys; r += stride) {
    int2 rc = make_int2(0, 0);
    if (!failed) {
      rc.x = a.root_cells[r].x;
      uint32_t nodes;
      rc.y = scan_children(a, rc.x, (uint32_t)a.off[r + 1], nodes);
      place_children(a, rc.x, rc.y, nodes);
    }
    a.root_cells[r] = rc;
  }
}

__global__ __launch_bounds__(kBlock) void k_cells_finish(LevelArgs a) {
  BT_BUILD_PRIO();
  if (blockIdx.x == 0) write_counters(a.dc, a.host);
  const int nc_all = a.dc->ncells;
  for (int s = blockIdx.x * kBlock + threadIdx.x; s < nc_all; s += gridDim.x * kBlock) {
    uint4 r = a.raw[s];
    const uint32_t L = r.x >> 27;
    r.x = (L == 1 ? 0u : (uint32_t)a.fin[r.x & 0x07FFFFFFu]) | (L << 27);
    const int f = a.fin[s];
    if (r.y != 0xFFFFFFFFu) {
      r.y = cell_pack_y((int)r.y, a.nch[s]);
      a.arrived[f] = 0;
    }
    a.cells[f] = r;
  }
}

// ---- bottom-up multipoles -------------------------------------------------

constexpr int kScrVecs = 5;   // vectors of a cell's scratch record

// T: the real type of particles and cell data (float or double).
template <typename T>
struct MpArgs {
  int L;
  T inv_theta;
  const V4<T> *pos;       // tree order
  const uint4 *cells;
  V4<T> *scr;             // 5 per cell: (ref,M) (com-ref,Qxz) (Qxx,Qyy,Qzz,Qxy) (bmin,Qyz) (bmax,-)
  V4<T> *size, *mono, *q0;
  V2<T> *q1, *ls;
  V4<T> *wrec;            // 3 per cell, the walk's P2C record
  int *arrived;           // per node: children whose records are written (zero before)
  const DevCounters *dc;
};

template <typename R>
struct Moments {
  R M, sx, sy, sz, xx, yy, zz, xy, xz, yz;
};

// The scratch record of a cell, which its parent's thread reads.  CLIMB: written
// and read by threads of one launch, so every access is an agent-scope atomic (it
// passes the XCD's own L2, which is not coherent with the others').
template <typename T, bool CLIMB>
__device__ __forceinline__ void scr_store(V4<T> *p, const V4<T> v) {
  if constexpr (CLIMB) {
    const unsigned long long *w = reinterpret_cast<const unsigned long long *>(&v);
#pragma unroll
    for (int k = 0; k < (int)(sizeof(v) / 8); k++)
      __hip_atomic_store(reinterpret_cast<unsigned long long *>(p) + k, w[k], __ATOMIC_RELAXED,
                         __HIP_MEMORY_SCOPE_AGENT);
  } else {
    *p = v;
  }
}
template <typename T, bool CLIMB>
__device__ __forceinline__ V4<T> scr_load(const V4<T> *p) {
  if constexpr (CLIMB) {
    V4<T> v;
    unsigned long long *w = reinterpret_cast<unsigned long long *>(&v);
#pragma unroll
    for (int k = 0; k < (int)(sizeof(v) / 8); k++)
      w[k] = __hip_atomic_load(reinterpret_cast<const unsigned long long *>(p) + k,
                               __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
    return v;
  } else {
    return *p;
  }
}

template <typename T, bool CLIMB>
__device__ void write_cell(const MpArgs<T> &a, int c, T rx, T ry, T rz, double M, double dx,
                           double dy, double dz, double qxx, double qyy, double qzz, double qxy,
                           double qxz, double qyz, const Ext<T> &e) {
#pragma clang fp contract(off)
  const T comx = (T)((double)rx + dx), comy = (T)((double)ry + dy), comz = (T)((double)rz + dz);
  const T bcx = (e.xx + e.nx) * T(0.5), bcy = (e.xy + e.ny) * T(0.5), bcz = (e.xz + e.nz) * T(0.5);
  const T hx = (e.xx - e.nx) * T(0.5), hy = (e.xy - e.ny) * T(0.5), hz = (e.xz - e.nz) * T(0.5);
  const T ex = bcx - comx, ey = bcy - comy, ez = bcz - comz;
  T s;
  if constexpr (sizeof(T) == 4) s = sqrtf(ex * ex + ey * ey + ez * ez);
  else s = sqrt(ex * ex + ey * ey + ez * ez);
  const T l = rmax(T(2) * rmax(hx, rmax(hy, hz)), T(1.0e-6));
  const T op = l * a.inv_theta + s;
  a.size[c] = make_v4<T>(comx, comy, comz, op * op);
  a.mono[c] = make_v4<T>(comx, comy, comz, (T)M);
  a.q0[c] = make_v4<T>((T)qxx, (T)qyy, (T)qzz, (T)qxy);
  a.q1[c] = make_v2<T>((T)qxz, (T)qyz);
  a.ls[c] = make_v2<T>(l, s);
  // walk record (p2c_rec): quadrupole pre-multiplied, trace terms precomputed
  const T fqxx = (T)qxx, fqyy = (T)qyy, fqzz = (T)qzz;
  const T tr = fqxx + fqyy + fqzz;
  a.wrec[3 * (size_t)c] = make_v4<T>(comx, comy, comz, (T)M);
  a.wrec[3 * (size_t)c + 1] = make_v4<T>(T(-7.5) * fqxx, T(-7.5) * fqyy, T(-7.5) * fqzz, T(-7.5) * (T)qxy);
  a.wrec[3 * (size_t)c + 2] =
      make_v4<T>(T(-7.5) * (T)qxz, T(-7.5) * (T)qyz, tr, T(1.5) * tr);
  V4<T> *rec = a.scr + kScrVecs * (size_t)c;
  scr_store<T, CLIMB>(rec, make_v4<T>(rx, ry, rz, (T)M));
  scr_store<T, CLIMB>(rec + 1, make_v4<T>((T)dx, (T)dy, (T)dz, (T)qxz));
  scr_store<T, CLIMB>(rec + 2, make_v4<T>((T)qxx, (T)qyy, (T)qzz, (T)qxy));
  scr_store<T, CLIMB>(rec + 3, make_v4<T>(e.nx, e.ny, e.nz, (T)qyz));
  scr_store<T, CLIMB>(rec + 4, make_v4<T>(e.xx, e.xy, e.xz, T(0)));
}

template <typename T, typename R, bool CLIMB>
__device__ void finish_moments(const MpArgs<T> &a, int c, T rx, T ry, T rz, const Moments<R> &m,
                               const Ext<T> &e) {
  if (!(m.M > R(0))) {
    write_cell<T, CLIMB>(a, c, rx, ry, rz, 0.0, 0, 0, 0, 0, 0, 0, 0, 0, 0, e);
    return;
  }
  const R im = R(1) / m.M;
  const R dx = m.sx * im, dy = m.sy * im, dz = m.sz * im;
  write_cell<T, CLIMB>(a, c, rx, ry, rz, (double)m.M, (double)dx, (double)dy, (double)dz,
                (double)(m.xx * im - dx * dx), (double)(m.yy * im - dy * dy),
                (double)(m.zz * im - dz * dz), (double)(m.xy * im - dx * dy),
                (double)(m.xz * im - dx * dz), (double)(m.yz * im - dy * dz), e);
}

template <typename T, typename R, bool CLIMB = false>
__device__ void node_moments(const MpArgs<T> &a, int c, const uint4 cd) {
  Moments<R> m{};
  Ext<T> e = ext_empty<T>();
  const int f = cell_first(cd), nc = cell_nchild(cd);
  struct Child {
    V4<T> g, d, q, bmn, bmx;
  };
  auto load = [&](int k) {
    const V4<T> *rec = a.scr + kScrVecs * (size_t)(f + k);
    return Child{scr_load<T, CLIMB>(rec), scr_load<T, CLIMB>(rec + 1), scr_load<T, CLIMB>(rec + 2),
                 scr_load<T, CLIMB>(rec + 3), scr_load<T, CLIMB>(rec + 4)};
  };
  // CLIMB: the records of kBatch children are in flight together (one at a time, with
  // the next loaded meanwhile, a node cost a latency per child: 57 -> 43 us at 2^16).
  // With many waves in flight, in the level launches, that only costs registers.
  constexpr int kBatch = !CLIMB ? 1 : sizeof(T) == 4 ? 8 : 4;
  V4<T> r0;   // this node's reference = first child's
  for (int k0 = 0; k0 < nc; k0 += kBatch) {
    Child child[kBatch];
#pragma unroll
    for (int q = 0; q < kBatch; q++) child[q] = load(min(k0 + q, nc - 1));
    if (k0 == 0) r0 = child[0].g;
#pragma unroll
    for (int q = 0; q < kBatch; q++) {
      if (k0 + q >= nc) break;
      const Child &ch = child[q];
      // child com relative to this node's reference: both references lie in the
      // node's bbox, so their difference is at most l and (near-)exact in T
      const R ox = R(ch.g.x - r0.x) + R(ch.d.x), oy = R(ch.g.y - r0.y) + R(ch.d.y),
              oz = R(ch.g.z - r0.z) + R(ch.d.z);
      const R Mc = R(ch.g.w);
      m.M += Mc;
      m.sx += Mc * ox; m.sy += Mc * oy; m.sz += Mc * oz;
      m.xx += Mc * (R(ch.q.x) + ox * ox); m.yy += Mc * (R(ch.q.y) + oy * oy);
      m.zz += Mc * (R(ch.q.z) + oz * oz); m.xy += Mc * (R(ch.q.w) + ox * oy);
      m.xz += Mc * (R(ch.d.w) + ox * oz); m.yz += Mc * (R(ch.bmn.w) + oy * oz);
      ext_merge(e, ch.bmn.x, ch.bmn.y, ch.bmn.z, ch.bmx.x, ch.bmx.y, ch.bmx.z);
    }
  }
  finish_moments<T, R, CLIMB>(a, c, r0.x, r0.y, r0.z, m, e);
}

// Treecode<float>: leaves sum in FP32, nodes combine in FP32 below level
// kFp64Levels and in FP64 at and above it.  Treecode<double>: FP64 throughout.
template <typename T, bool CLIMB = false>
__device__ __forceinline__ void leaf_moments(const MpArgs<T> &a, int c, const uint4 cd) {
  const int pb = (int)cd.z, pe = (int)cd.w;
  Moments<T> m{};
  Ext<T> e = ext_empty<T>();
  const V4<T> r0 = a.pos[pb];  // reference point: the first particle
  auto add = [&](const V4<T> p) {
    ext_add(e, p.x, p.y, p.z);
    const T dx = p.x - r0.x, dy = p.y - r0.y, dz = p.z - r0.z, w = p.w;
    m.M += w;
    m.sx += w * dx; m.sy += w * dy; m.sz += w * dz;
    m.xx += w * dx * dx; m.yy += w * dy * dy; m.zz += w * dz * dz;
    m.xy += w * dx * dy; m.xz += w * dx * dz; m.yz += w * dy * dz;
  };
  // particles in order, the loads of kBatch issued together; CLIMB: those past the end
  // too (of the last particle), as few waves hide a remainder's latencies
  constexpr int kBatch = !CLIMB ? 4 : sizeof(T) == 4 ? 16 : 8;
  int i = pb;
  for (; CLIMB ? i < pe : i + kBatch <= pe; i += kBatch) {
    V4<T> p[kBatch];
#pragma unroll
    for (int q = 0; q < kBatch; q++) p[q] = a.pos[CLIMB ? min(i + q, pe - 1) : i + q];
#pragma unroll
    for (int q = 0; q < kBatch; q++)
      if (!CLIMB || i + q < pe) add(p[q]);
  }
  for (; i < pe; i++) add(a.pos[i]);
  finish_moments<T, T, CLIMB>(a, c, r0.x, r0.y, r0.z, m, e);
}

// The cells of one level, whose children are done.  (The leaves of all levels in a
// launch of their own: 0.74 ms against 0.67 at 2^24 particles, as the cell arrays'
// lines are then written in parts.)
template <typename T, typename R>
__global__ __launch_bounds__(kBlock) void k_multipole_level(MpArgs<T> a) {
  BT_BUILD_PRIO();
  const int cnt = a.dc->lvl_count[a.L];
  const int c0 = a.dc->lvl_start[a.L];
  for (int t = blockIdx.x * kBlock + threadIdx.x; t < cnt; t += gridDim.x * kBlock) {
    const uint4 cd = a.cells[c0 + t];
    if (cell_leaf(cd)) leaf_moments<T>(a, c0 + t, cd);
    else node_moments<T, R>(a, c0 + t, cd);
  }
}

// All cells of a small tree in one launch: the thread of a leaf climbs.  At each
// parent it counts itself in; the last child to arrive combines the parent's
// children (in their order, so the result does not depend on who arrives last) and
// goes on from there.  Nothing waits.  The count of a parent is raised only after
// the stores of the child's record have completed, and its children's records are
// read after the count has shown them all: both by agent-scope accesses.
//
// Each of these accesses is coherent over the chip by itself; their order is gfx950's,
// not the language's: the stores have been made when vmcnt is 0, and the loads of the
// records are issued after the add, on whose result they depend, has returned.  (The
// cells and the zeroed counts are a launch older.)  A release fence before the add and an
// acquire fence after it would say so in the language, but write back and invalidate
// whole caches in every step of every wave: 67 -> 136 us at 3*10^5 particles, 103 -> 274
// at 7*10^5.  For another target, or for records that are not read and written by such
// accesses, they are needed.
template <typename T>
__global__ __launch_bounds__(kBlock) void k_multipole_climb(MpArgs<T> a) {
  BT_BUILD_PRIO();
  const int ncells = a.dc->ncells;
  for (int t = blockIdx.x * kBlock + threadIdx.x; t < ncells; t += gridDim.x * kBlock) {
    int c = t;
    uint4 cd = a.cells[c];
    if (!cell_leaf(cd)) continue;
    leaf_moments<T, true>(a, c, cd);
    for (int L = (int)(cd.x >> 27); L > 1; L--) {
      asm volatile("s_waitcnt vmcnt(0)" ::: "memory");   // this cell's record is out
      const int p = (int)(cd.x & 0x07FFFFFFu);
      cd = a.cells[p];
      const int before = __hip_atomic_fetch_add(a.arrived + p, 1, __ATOMIC_RELAXED,
                                                __HIP_MEMORY_SCOPE_AGENT);
      if (before + 1 < cell_nchild(cd)) break;
      __hip_atomic_store(a.arrived + p, 0, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);  // for the next call
      c = p;
      if (sizeof(T) == 8 || L - 1 <= kFp64Levels) node_moments<T, double, true>(a, c, cd);
      else node_moments<T, float, true>(a, c, cd);
    }
  }
}

}  // namespace

namespace {

bool box_with_keys(const Ctx &c) { return c.nsys == 1 && c.bbox_blocks <= kBoxParts; }

template <typename R>
void bbox_t(Ctx &c) {
  const int nb = c.bbox_blocks;
  hipLaunchKernelGGL(k_bbox_partial<R>, dim3(nb, c.nsys), dim3(kBlock), 0, c.stream, as4<R>(c.pos),
                     c.d_off, nb, as4<R>(c.bbox_part));
  if (box_with_keys(c)) return;
  hipLaunchKernelGGL(k_bbox_final<R>, dim3(c.nsys), dim3(kBlock), 0, c.stream,
                     as4<R>(c.bbox_part), nb, as4<R>(c.box));
}

template <typename R>
void geo_keys_t(Ctx &c) {
  auto kern = box_with_keys(c) ? k_geo_keys<R, true> : k_geo_keys<R, false>;
  hipLaunchKernelGGL(kern, dim3(grid_for(c.n, kBlock, 8192)), dim3(kBlock), 0, c.stream, c.n,
                     c.nsys, c.d_off, as4<R>(c.box), as4<R>(c.bbox_part), c.bbox_blocks,
                     as4<R>(c.pos), c.geo_keys, c.valA, c.dc);
}

}  // namespace

void launch_bbox(Ctx &c) {
  if (c.fp64) bbox_t<double>(c);
  else bbox_t<float>(c);
}

// After launch_bbox, which may have left the box to this launch.
void launch_geo_keys(Ctx &c) {
  if (c.fp64) geo_keys_t<double>(c);
  else geo_keys_t<float>(c);
}

namespace {

template <typename T>
auto gather_kernel(bool is_short, bool forest, bool ident) {
  if (!is_short) return ident ? k_gather3<T, false, false, true> : k_gather3<T, false, false, false>;
  if (forest) return ident ? k_gather3<T, true, true, true> : k_gather3<T, true, true, false>;
  return ident ? k_gather3<T, true, false, true> : k_gather3<T, true, false, false>;
}

}  // namespace

void launch_gather_tree(Ctx &c) {
  const dim3 g(grid_for(c.n, kBlock, 8192));
  const bool is_short = c.geo_low > 0, forest = c.nsys > 1;
  const int *perm = is_short ? c.valB : c.valA;
  if (c.fp64)
    hipLaunchKernelGGL(gather_kernel<double4>(is_short, forest, c.ids_in_order), g, dim3(kBlock), 0,
                       c.stream, c.n, perm, as4<double>(c.pos), as4<double>(c.vel), c.id,
                       as4<double>(c.pos2), as4<double>(c.vel2), c.id2, c.geo_low, c.keyB,
                       c.geo_keys, c.nsys, c.d_off, c.dc);
  else
    hipLaunchKernelGGL(gather_kernel<float4>(is_short, forest, c.ids_in_order), g, dim3(kBlock), 0,
                       c.stream, c.n, perm, c.pos, c.vel, c.id, c.pos2, c.vel2, c.id2, c.geo_low,
                       c.keyB, c.geo_keys, c.nsys, c.d_off, c.dc);
  c.ids_in_order = false;
  std::swap(c.pos, c.pos2);
  std::swap(c.vel, c.vel2);
  std::swap(c.id, c.id2);
}

int cell_tiles(int n) {   // particle n, past the last, included
  return n / (kBlock * (n <= kCellSmall ? 1 : kCellRounds)) + 1;
}

// the most tiles that any number of particles up to n takes
int max_cell_tiles(int n) { return std::max(cell_tiles(n), cell_tiles(std::min(n, kCellSmall))); }

void launch_levels(Ctx &c, bool read) {
  LevelArgs a;
  a.nsys = c.nsys;
  a.nleaf = c.nleaf;
  a.cap_cells = c.cap_cells;
  a.n = c.n;
  a.ntiles = cell_tiles(c.n);
  a.off = c.d_off;
  a.keys = c.geo_keys;
  a.cells = c.cells;
  a.raw = c.cell_raw;
  a.fin = c.cell_fin;
  a.nch = c.cell_nch;
  a.arrived = c.cell_arrived;
  a.cnt = c.cell_cnt;
  a.root_cells = c.root_cells;
  a.level_beg = c.level_beg;
  a.dc = c.dc;
  a.host = read ? c.pinned_dc : nullptr;
  const dim3 tiles(a.ntiles), cells(grid_for(std::max(c.cap_cells, c.nsys), kBlock, 4096));
  const bool forest = c.nsys > 1;
  const bool small = c.n <= kCellSmall;
  auto count = small ? (forest ? k_cells_count<true, 1> : k_cells_count<false, 1>)
                     : (forest ? k_cells_count<true, kCellRounds> : k_cells_count<false, kCellRounds>);
  auto emit = small ? (forest ? k_cells_emit<true, 1> : k_cells_emit<false, 1>)
                    : (forest ? k_cells_emit<true, kCellRounds> : k_cells_emit<false, kCellRounds>);
  hipLaunchKernelGGL(count, tiles, dim3(kBlock), 0, c.stream, a);
  hipLaunchKernelGGL(k_cells_scan, dim3(kCellRows), dim3(kScanBlock), 0, c.stream, a);
  hipLaunchKernelGGL(emit, tiles, dim3(kBlock), 0, c.stream, a);
  hipLaunchKernelGGL(k_cells_place, cells, dim3(kBlock), 0, c.stream, a);
  hipLaunchKernelGGL(k_cells_finish, cells, dim3(kBlock), 0, c.stream, a);
}

namespace {

template <typename T>
void multipoles_t(Ctx &c) {
  MpArgs<T> a;
  a.inv_theta = (T)(1.0 / (double)c.theta);
  a.pos = as4<T>(c.pos);
  a.cells = c.cells;
  a.scr = as4<T>(c.cscr);
  a.size = as4<T>(c.csize);
  a.mono = as4<T>(c.cmono);
  a.q0 = as4<T>(c.cq0);
  a.q1 = as2<T>(c.cq1);
  a.ls = as2<T>(c.cls);
  a.wrec = as4<T>(c.cwalk);
  a.arrived = c.cell_arrived;
  a.dc = c.dc;
  const int grid = grid_for(c.cap_cells, kBlock, 2048);
  // computeMultipoles, one launch per level / one in all: 2^16 88 / 43 us, 4*10^5 140 /
  // 86, 7*10^5 150 / 120, 10^6 159 / 148, 2*10^6 175 / 243 (records past the L2 cost more
  // than launches); FP64 4*10^5 175 / 138
  if (c.n <= 1 << 20) {
    hipLaunchKernelGGL(k_multipole_climb<T>, dim3(grid), dim3(kBlock), 0, c.stream, a);
    return;
  }
  for (int L = kMaxLevel; L >= 1; L--) {
    a.L = L;
    auto kern = sizeof(T) == 8 || L <= kFp64Levels ? k_multipole_level<T, double>
                                                   : k_multipole_level<T, T>;
    hipLaunchKernelGGL(kern, dim3(grid), dim3(kBlock), 0, c.stream, a);
  }
}

}  // namespace

void launch_multipoles(Ctx &c) {
  if (c.fp64) multipoles_t<double>(c);
  else multipoles_t<float>(c);
}

}  // namespace bt
