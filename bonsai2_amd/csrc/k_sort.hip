// k_sort.hip -- stable LSD radix sort of (u64 key, int value) pairs and
// device-wide scans, written for wave64.
//
// Replaces thrust::sort_by_key / thrust::inclusive_scan_by_key of the
// reference (code/makeGroups.cu:270-295, code/buildTree.cu:940-944), whose
// contract is kept: nondecreasing keys, ties in input order.
//
// One pass = 8-bit digit: (1) per-tile histograms in LDS, written digit-major;
// (2) exclusive scan of each digit's row over the tiles, one block per digit, and the
// digits' totals, which the scatter's blocks scan themselves (one launch; a scan of the
// whole array took two, 9 us instead of 3 at 10^6 pairs, 12 instead of 6 at 2*10^7);
// (3) stable ranks: each wave ranks its contiguous eighth of the tile with 8
// ballots per 64 pairs (lanes with equal digits form a peer mask) against its
// own digit counters in LDS, keeping the pairs in registers; the waves' counts
// are then chained per digit, each pair is placed at its sorted position
// within the tile in LDS, and the tile is written out in that order, so
// consecutive threads store consecutive addresses of one digit's run (whole
// cache lines instead of one scattered store per pair).
// A tile is 512 threads x 8 rounds = 4096 pairs; HBM traffic per pass is
// ~8 B (histogram read) + 12 B read + 12 B written per pair.  Up to 2^17 pairs of one
// system are sorted by tiles in LDS and merged instead (below).
#include "bt_device.h"
#include "bt_internal.h"

namespace bt {

namespace {

constexpr int kSortThreads = 256;
constexpr int kSortRounds = 16;
constexpr int kSortTile = kSortThreads * kSortRounds;
// The three-launch passes run the same 4096-pair tile with 512 threads (8
// waves of 8 rounds): twice the waves per CU for the same LDS.
constexpr int kCThreads = 512;
constexpr int kCRounds = kSortTile / kCThreads;
constexpr int kCWaves = kCThreads / kWave;
static_assert(kCThreads * kCRounds == kSortTile, "tile of the three-launch passes");
constexpr int kScanThreads = 256;
constexpr int kScanItems = 8;
constexpr int kScanTile = kScanThreads * kScanItems;
// up to this many tiles a scan takes two launches (the down-sweep reduces the
// tile totals before it, at most 1024 ints per block); beyond, three
constexpr int kScanFusedTiles = 1024;

struct DigitSrc {
  int shift;        // bit offset of the digit
  int nsys;
  const int *off;
};

// BYSYS: the digit is taken from system_of(value) instead of the key (a
// compile-time choice, so the key passes carry no branch and their loads can
// all be issued before the first is used).
template <bool BYSYS>
__device__ __forceinline__ int digit_of(uint64_t key, int val, const DigitSrc &s) {
  if (BYSYS) return (system_of(val, s.nsys, s.off) >> s.shift) & 0xFF;
  return (int)((key >> s.shift) & 0xFFull);
}

// ---- scans ---------------------------------------------------------------

struct OpSum {
  static __device__ __forceinline__ int id() { return 0; }
  static __device__ __forceinline__ int op(int a, int b) { return a + b; }
};

// Inclusive scan across a 256-thread block; returns inclusive value, *total = block total.
template <class Op>
__device__ __forceinline__ int block_incl_scan(int v, int *sh_wave, int *total) {
  const int l = lane_id(), w = threadIdx.x >> 6;
#pragma unroll
  for (int d = 1; d < kWave; d <<= 1) {
    const int t = __shfl_up(v, d, kWave);
    if (l >= d) v = Op::op(t, v);
  }
  if (l == kWave - 1) sh_wave[w] = v;
  __syncthreads();
  int pre = Op::id();
  for (int k = 0; k < w; k++) pre = Op::op(pre, sh_wave[k]);
  int tot = Op::id();
  for (int k = 0; k < (int)(blockDim.x >> 6); k++) tot = Op::op(tot, sh_wave[k]);
  *total = tot;
  __syncthreads();
  return Op::op(pre, v);
}

template <bool BYSYS>
__global__ __launch_bounds__(kCThreads) void k_radix_hist(const uint64_t *__restrict__ keys,
                                                          const int *__restrict__ vals,
                                                          int n, DigitSrc src, int nblocks,
                                                          int *__restrict__ ghist) {
  BT_BUILD_PRIO();
  __shared__ int hist[256];
  const int tid = threadIdx.x;
  if (tid < 256) hist[tid] = 0;
  const int base = blockIdx.x * kSortTile;
  // all of the tile's loads first, then the LDS counting
  int dg[kCRounds];
#pragma unroll
  for (int r = 0; r < kCRounds; r++) {
    const int i = base + r * kCThreads + tid;
    const int ic = min(i, n - 1);   // unconditional loads: no branch between them
    const int d = digit_of<BYSYS>(BYSYS ? 0ull : keys[ic], BYSYS ? vals[ic] : 0, src);
    dg[r] = i < n ? d : -1;
  }
  __syncthreads();
#pragma unroll
  for (int r = 0; r < kCRounds; r++)
    if (dg[r] >= 0) atomicAdd(&hist[dg[r]], 1);
  __syncthreads();
  if (tid < 256) ghist[tid * nblocks + blockIdx.x] = hist[tid];
}

// Block d: row d of the histogram to its exclusive prefix over the tiles, the total to
// total[d].
constexpr int kRowThreads = 512, kRowPer = 4;
__global__ __launch_bounds__(kRowThreads) void k_radix_rows(int nblocks, int *__restrict__ ghist,
                                                            int *__restrict__ total) {
  BT_BUILD_PRIO();
  __shared__ int shw[kRowThreads / kWave];
  int *row = ghist + (size_t)blockIdx.x * nblocks;
  const int w = threadIdx.x >> 6;
  int carry = 0;
  for (int b0 = 0; b0 < nblocks; b0 += kRowThreads * kRowPer) {
    int v[kRowPer], own = 0;
    const int i0 = b0 + threadIdx.x * kRowPer;
#pragma unroll
    for (int k = 0; k < kRowPer; k++) {
      v[k] = i0 + k < nblocks ? row[i0 + k] : 0;
      own += v[k];
    }
    const int incl = wave_incl_scan(own);
    if (lane_id() == kWave - 1) shw[w] = incl;
    __syncthreads();
    int run = carry + incl - own;
#pragma unroll
    for (int k = 0; k < kRowThreads / kWave; k++) {
      run += k < w ? shw[k] : 0;
      carry += shw[k];
    }
#pragma unroll
    for (int k = 0; k < kRowPer; k++) {
      if (i0 + k < nblocks) row[i0 + k] = run;
      run += v[k];
    }
    __syncthreads();
  }
  if (threadIdx.x == 0) total[blockIdx.x] = carry;
}

template <bool BYSYS>
__global__ __launch_bounds__(kCThreads) void k_radix_scatter(
    const uint64_t *__restrict__ keys, const int *__restrict__ vals, int n, DigitSrc src,
    int nblocks, const int *__restrict__ goff, const int *__restrict__ total,
    uint64_t *__restrict__ keys_out, int *__restrict__ vals_out) {
  BT_BUILD_PRIO();
  // LDS kept under a third of a CU's 160 KiB, so three blocks share a CU:
  // 16-bit per-wave digit counters (a tile holds 4096 pairs) and, per digit,
  // only (global base - tile-local start)
  __shared__ uint64_t skeys[kSortTile];   // the tile in sorted order
  __shared__ int svals[kSortTile];
  __shared__ int gdelta[256];     // global position of digit d's pairs minus their tile start
  __shared__ unsigned short wcnt[kCWaves][256];   // per-wave digit counts -> digit bases
  __shared__ int sh_cnt[kCWaves], sh_tot[kCWaves];
  const int tid = threadIdx.x;
  const int w = tid >> 6;
  const int lane = lane_id();
  int tstart = 0;   // thread d < 256: first tile-local position of digit d
  {
    // thread d < 256: digit d's pairs in the tiles before, in this tile and in all
    int g0 = 0, cnt = 0, tot = 0;
    if (tid < 256) {
      const int *row = goff + (size_t)tid * nblocks + blockIdx.x;
      g0 = row[0];
      tot = total[tid];
      cnt = ((int)blockIdx.x + 1 < nblocks ? row[1] : tot) - g0;
    }
    const int icnt = wave_incl_scan(cnt), itot = wave_incl_scan(tot);
    if (lane == kWave - 1) {
      sh_cnt[w] = icnt;
      sh_tot[w] = itot;
    }
    __syncthreads();
    tstart = icnt - cnt;
    int gstart = itot - tot;
    for (int k = 0; k < 256 / kWave; k++) {
      tstart += k < w ? sh_cnt[k] : 0;
      gstart += k < w ? sh_tot[k] : 0;
    }
    if (tid < 256) gdelta[tid] = gstart + g0 - tstart;
  }
  for (int k = tid; k < kCWaves * 256; k += kCThreads) (&wcnt[0][0])[k] = 0;
  __syncthreads();
  // Each wave ranks its own contiguous eighth of the tile (8 rounds of 64
  // pairs) against its private digit counters; pairs stay in registers.
  const int wbase = blockIdx.x * kSortTile + w * (kCRounds * kWave);
  uint64_t kk[kCRounds];
  int vv[kCRounds], dd[kCRounds], rr[kCRounds];
  // the wave's rounds of pairs are all loaded before the ranking starts
#pragma unroll
  for (int r = 0; r < kCRounds; r++) {
    const int i = wbase + r * kWave + lane;
    kk[r] = i < n ? keys[i] : 0ull;
    vv[r] = i < n ? vals[i] : 0;
  }
#pragma unroll
  for (int r = 0; r < kCRounds; r++) {
    const int i = wbase + r * kWave + lane;
    const bool valid = i < n;
    const uint64_t key = kk[r];
    const int val = vv[r];
    const int d = valid ? digit_of<BYSYS>(key, val, src) : 0;
    const uint64_t peers = same_digit(ballot64(valid), d);
    const int rank = lanes_before(peers);
    const int before = wcnt[w][d];
    wave_lds_sync();
    if (valid && rank == 0) wcnt[w][d] = (unsigned short)(before + __popcll(peers));
    wave_lds_sync();
    dd[r] = valid ? d : -1;
    rr[r] = before + rank;
  }
  __syncthreads();
  if (tid < 256) {
    // digit tid: the waves' pairs follow each other in tile order
    int acc = tstart;
#pragma unroll
    for (int k = 0; k < kCWaves; k++) {
      const int c = wcnt[k][tid];
      wcnt[k][tid] = (unsigned short)acc;
      acc += c;
    }
  }
  __syncthreads();
#pragma unroll
  for (int r = 0; r < kCRounds; r++) {
    if (dd[r] >= 0) {
      const int pos = wcnt[w][dd[r]] + rr[r];
      skeys[pos] = kk[r];
      svals[pos] = vv[r];
    }
  }
  __syncthreads();
  const int base = blockIdx.x * kSortTile;
  const int tile_n = min(kSortTile, n - base);
  for (int j = tid; j < tile_n; j += kCThreads) {
    const uint64_t key = skeys[j];
    const int val = svals[j];
    const int d = digit_of<BYSYS>(key, val, src);
    const int dst = gdelta[d] + j;
    keys_out[dst] = key;
    vals_out[dst] = val;
  }
}

// ---- one-sweep passes ------------------------------------------------------
// The digit counts of every pass come from one histogram launch over the
// input (the digits of a key do not change while it moves between passes).
// Each pass is then one launch: a block takes the next tile from a counter,
// ranks its pairs as above, publishes its per-digit counts and finds the
// counts of all earlier tiles by looking back through their status words
// (decoupled look-back), then writes its pairs to their sorted positions.
// Per pass: 12 B read + 12 B written per pair.
//
// A status word is (flag << 30) | count, flag 1 = this tile's count only,
// 2 = the inclusive count of tiles 0..t.  A block waits only for tiles that
// were handed out before its own, whose blocks are already running and never
// wait for later tiles, so the wait ends; it is bounded anyway and reports
// kSortErr instead of hanging.  Two status buffers and two tile counters
// alternate between passes: a pass clears the other buffer's words of its
// tile and resets the other counter for the next pass.

constexpr int kMaxSortPasses = 11;
// One-sweep tiles: 256 threads x 8 rounds = 2048 pairs (30 KiB of LDS, so
// five blocks share a CU while others wait in their look-back).
constexpr int kOsRounds = 8;
constexpr int kOsTile = kSortThreads * kOsRounds;
constexpr int kSortHistBlocks = 1024;
constexpr unsigned kStAgg = 1u << 30, kStIncl = 2u << 30, kStCount = (1u << 30) - 1u;
constexpr int kLookbackSpins = 1 << 22;

struct PassSet {
  int np;
  int nsys;
  const int *off;
  int shift[kMaxSortPasses];
  int bysys[kMaxSortPasses];
};

// Adds 1 for every valid lane at hist[d].  A wave whose valid lanes all hold
// one digit (the high digits of nearly sorted keys) adds its count with one
// atomic; otherwise each lane adds its own.
__device__ __forceinline__ void wave_count_digit(int *hist, int d, bool valid) {
  const uint64_t vm = ballot64(valid);
  if (vm == 0) return;   // wave-uniform
  const int first = __ffsll((unsigned long long)vm) - 1;
  const int d0 = __shfl(d, first, kWave);
  const uint64_t same = ballot64(valid && d == d0);
  if (same == vm) {
    if (lane_id() == first) atomicAdd(&hist[d0], __popcll(vm));
  } else if (valid) {
    atomicAdd(&hist[d], 1);
  }
}

// grid kSortHistBlocks: block b counts the digits of every pass over a
// contiguous chunk; part[b][p][256].
__global__ __launch_bounds__(kSortThreads) void k_radix_hist_all(const uint64_t *__restrict__ keys,
                                                                 const int *__restrict__ vals,
                                                                 int n, PassSet ps,
                                                                 int *__restrict__ part,
                                                                 DevCounters *dc) {
  __shared__ int hist[kMaxSortPasses * 256];
  // the sort error bit reports this sort only (err_sticky keeps it for the step)
  if (blockIdx.x == 0 && threadIdx.x == 0) atomicAnd(&dc->err, ~kSortErr);
  for (int k = threadIdx.x; k < ps.np * 256; k += kSortThreads) hist[k] = 0;
  __syncthreads();
  const int chunk = (n + gridDim.x - 1) / gridDim.x;
  const int i0 = blockIdx.x * chunk, i1 = min(n, i0 + chunk);
  for (int j0 = i0; j0 < i1; j0 += kSortThreads) {
    const int i = j0 + threadIdx.x;
    const bool valid = i < i1;
    const uint64_t key = valid ? keys[i] : 0ull;
    const int val = valid ? vals[i] : 0;
    for (int p = 0; p < ps.np; p++) {
      const DigitSrc src{ps.shift[p], ps.nsys, ps.off};
      const int d = ps.bysys[p] ? digit_of<true>(key, val, src) : digit_of<false>(key, val, src);
      wave_count_digit(hist + p * 256, d, valid);
    }
  }
  __syncthreads();
  for (int k = threadIdx.x; k < ps.np * 256; k += kSortThreads)
    part[(size_t)blockIdx.x * ps.np * 256 + k] = hist[k];
}

// grid (passes, 8): block (p, g) sums digits [32g, 32g + 32) of pass p over
// the histogram blocks, 8 segments of blocks per digit in parallel.
__global__ __launch_bounds__(256) void k_radix_hist_sum(const int *__restrict__ part, int np,
                                                        int nparts, int *__restrict__ gcount) {
  __shared__ int sh[8][32];
  const int p = blockIdx.x;
  const int d = blockIdx.y * 32 + (threadIdx.x & 31);
  const int seg = threadIdx.x >> 5;
  const int per = (nparts + 7) / 8;
  const int b0 = seg * per, b1 = min(nparts, b0 + per);
  int s = 0;
#pragma unroll 8
  for (int b = b0; b < b1; b++) s += part[(size_t)b * np * 256 + p * 256 + d];
  sh[seg][threadIdx.x & 31] = s;
  __syncthreads();
  if (threadIdx.x < 32) {
    int t = 0;
    for (int k = 0; k < 8; k++) t += sh[k][threadIdx.x];
    gcount[p * 256 + d] = t;
  }
}

template <bool BYSYS>
__global__ __launch_bounds__(kSortThreads) void k_radix_onesweep(
    const uint64_t *__restrict__ keys, const int *__restrict__ vals, int n, DigitSrc src,
    const int *__restrict__ gcount, unsigned int *status, unsigned int *status_next, int *ctr,
    int *ctr_next, int ntiles, DevCounters *dc, uint64_t *__restrict__ keys_out,
    int *__restrict__ vals_out) {
  __shared__ uint64_t skeys[kOsTile];   // the tile in sorted order
  __shared__ int svals[kOsTile];
  __shared__ int tstart[256];     // first tile-local position of each digit
  __shared__ int gbase[256];      // global position of this tile's first pair of each digit
  __shared__ int wcnt[4][256];    // per-wave digit counts -> per-wave digit bases
  __shared__ int sh_wave[4];
  __shared__ int s_tile;
  const int tid = threadIdx.x;
  const int w = tid >> 6;
  const int lane = lane_id();
  if (tid == 0) s_tile = atomicAdd(ctr, 1);
#pragma unroll
  for (int k = 0; k < 4; k++) wcnt[k][tid] = 0;
  __syncthreads();
  const int tile = s_tile;
  if (tile >= ntiles) {   // a counter not reset: never index past the status words
    if (tid == 0) {
      atomicOr(&dc->err, kSortErr);
      atomicOr(&dc->err_sticky, kSortErr);
    }
    return;
  }
  if (tile == 0 && tid == 0) *ctr_next = 0;
  status_next[(size_t)tile * 256 + tid] = 0u;
  // Each wave ranks its own contiguous quarter of the tile (16 rounds of 64
  // pairs) against its private digit counters; pairs stay in registers.
  const int wbase = tile * kOsTile + w * (kOsRounds * kWave);
  uint64_t kk[kOsRounds];
  int vv[kOsRounds], dd[kOsRounds], rr[kOsRounds];
#pragma unroll
  for (int r = 0; r < kOsRounds; r++) {
    const int i = wbase + r * kWave + lane;
    kk[r] = i < n ? keys[i] : 0ull;
    vv[r] = i < n ? vals[i] : 0;
  }
#pragma unroll
  for (int r = 0; r < kOsRounds; r++) {
    const int i = wbase + r * kWave + lane;
    const bool valid = i < n;
    const int d = valid ? digit_of<BYSYS>(kk[r], vv[r], src) : 0;
    const uint64_t peers = same_digit(ballot64(valid), d);
    const int rank = lanes_before(peers);
    const int before = wcnt[w][d];
    wave_lds_sync();
    if (valid && rank == 0) wcnt[w][d] = before + __popcll(peers);
    wave_lds_sync();
    dd[r] = valid ? d : -1;
    rr[r] = before + rank;
  }
  __syncthreads();
  // digit tid: this tile's count, published before anything else is done
  const int cnt = wcnt[0][tid] + wcnt[1][tid] + wcnt[2][tid] + wcnt[3][tid];
  unsigned int *mine = status + (size_t)tile * 256 + tid;
  __hip_atomic_store(mine, (tile == 0 ? kStIncl : kStAgg) | (unsigned)cnt, __ATOMIC_RELAXED,
                     __HIP_MEMORY_SCOPE_AGENT);
  // tile-local start of each digit, and the global start of each digit
  int tot;
  const int incl = block_incl_scan<OpSum>(cnt, sh_wave, &tot);
  tstart[tid] = incl - cnt;
  const int g = gcount[tid];
  const int gincl = block_incl_scan<OpSum>(g, sh_wave, &tot);
  // look back over the earlier tiles until one holds an inclusive count
  int excl = 0;
  if (tile > 0) {
    int j = tile - 1;
    int spins = 0;
    for (;;) {
      const unsigned v = __hip_atomic_load(status + (size_t)j * 256 + tid, __ATOMIC_RELAXED,
                                           __HIP_MEMORY_SCOPE_AGENT);
      if ((v & ~kStCount) == 0u) {
        if (++spins > kLookbackSpins) {
          atomicOr(&dc->err, kSortErr);
          atomicOr(&dc->err_sticky, kSortErr);
          break;
        }
        __builtin_amdgcn_s_sleep(1);
        continue;
      }
      excl += (int)(v & kStCount);
      if ((v & ~kStCount) == kStIncl || j == 0) break;
      j--;
    }
    __hip_atomic_store(mine, kStIncl | (unsigned)(excl + cnt), __ATOMIC_RELAXED,
                       __HIP_MEMORY_SCOPE_AGENT);
  }
  gbase[tid] = gincl - g + excl;
  {
    // digit tid: the waves' pairs follow each other in tile order
    int acc = tstart[tid];
#pragma unroll
    for (int k = 0; k < 4; k++) {
      const int c = wcnt[k][tid];
      wcnt[k][tid] = acc;
      acc += c;
    }
  }
  __syncthreads();
#pragma unroll
  for (int r = 0; r < kOsRounds; r++) {
    if (dd[r] >= 0) {
      const int pos = wcnt[w][dd[r]] + rr[r];
      skeys[pos] = kk[r];
      svals[pos] = vv[r];
    }
  }
  __syncthreads();
  const int tile_n = min(kOsTile, n - tile * kOsTile);
  for (int j = tid; j < tile_n; j += kSortThreads) {
    const uint64_t key = skeys[j];
    const int val = svals[j];
    const int d = digit_of<BYSYS>(key, val, src);
    const int dst = gbase[d] + (j - tstart[d]);
    keys_out[dst] = key;
    vals_out[dst] = val;
  }
}

__global__ void k_sort_clear(unsigned int *status, int nwords, int *ctr) {
  for (int i = blockIdx.x * blockDim.x + threadIdx.x; i < nwords; i += gridDim.x * blockDim.x)
    status[i] = 0u;
  if (blockIdx.x == 0 && threadIdx.x == 0) *ctr = 0;
}


template <class Op>
__global__ __launch_bounds__(kScanThreads) void k_scan_reduce(const int *__restrict__ in, int n,
                                                              int *__restrict__ blk) {
  BT_BUILD_PRIO();
  __shared__ int shw[4];
  const int base = blockIdx.x * kScanTile;
  int v = Op::id();
#pragma unroll
  for (int k = 0; k < kScanItems; k++) {
    const int i = base + k * kScanThreads + threadIdx.x;
    if (i < n) v = Op::op(v, in[i]);
  }
  int total;
  block_incl_scan<Op>(v, shw, &total);
  if (threadIdx.x == 0) blk[blockIdx.x] = total;
}

// Exclusive scan of the block totals in place (one block, any count).
template <class Op>
__global__ __launch_bounds__(kScanThreads) void k_scan_blocks(int *__restrict__ blk, int nb,
                                                              int *__restrict__ total_dev) {
  BT_BUILD_PRIO();
  __shared__ int shw[4];
  int carry = Op::id();
  for (int b0 = 0; b0 < nb; b0 += kScanThreads) {
    const int i = b0 + threadIdx.x;
    const int v = i < nb ? blk[i] : Op::id();
    int total;
    const int inc = block_incl_scan<Op>(v, shw, &total);
    // exclusive = inclusive of the previous lane
    int exc = __shfl_up(inc, 1, kWave);
    const int w = threadIdx.x >> 6;
    if (lane_id() == 0) {
      exc = Op::id();
      for (int k = 0; k < w; k++) exc = Op::op(exc, shw[k]);
    }
    __syncthreads();
    if (i < nb) blk[i] = Op::op(carry, exc);
    carry = Op::op(carry, total);
    __syncthreads();
  }
  if (threadIdx.x == 0 && total_dev) *total_dev = carry;
}

// kPrefix: blk holds the tile totals and each block reduces those of the
// tiles before it itself (for few tiles: one launch instead of a separate
// scan of the totals); the last block writes the grand total to total_dev.
// Otherwise blk holds the tiles' exclusive prefixes (k_scan_blocks).
template <class Op, bool kPrefix>
__global__ __launch_bounds__(kScanThreads) void k_scan_down(const int *__restrict__ in, int n,
                                                            const int *__restrict__ blk,
                                                            int *__restrict__ out,
                                                            int *__restrict__ total_dev) {
  BT_BUILD_PRIO();
  __shared__ int sh[kScanTile];
  __shared__ int shw[4];
  const int base = blockIdx.x * kScanTile;
  int prefix;
  if constexpr (kPrefix) {
    int v = Op::id();
    for (int k = threadIdx.x; k < (int)blockIdx.x; k += kScanThreads) v = Op::op(v, blk[k]);
    (void)block_incl_scan<Op>(v, shw, &prefix);   // prefix = the reduction over the block
  } else {
    prefix = blk[blockIdx.x];
  }
#pragma unroll
  for (int k = 0; k < kScanItems; k++) {
    const int i = base + k * kScanThreads + threadIdx.x;
    sh[k * kScanThreads + threadIdx.x] = i < n ? in[i] : Op::id();
  }
  __syncthreads();
  // thread t owns items [t*8, t*8+8) of the tile
  int vals[kScanItems];
  int run = Op::id();
#pragma unroll
  for (int k = 0; k < kScanItems; k++) {
    vals[k] = sh[threadIdx.x * kScanItems + k];
    run = Op::op(run, vals[k]);
  }
  int total;
  const int inc = block_incl_scan<Op>(run, shw, &total);
  int exc = __shfl_up(inc, 1, kWave);
  if (lane_id() == 0) {
    exc = Op::id();
    const int w = threadIdx.x >> 6;
    for (int k = 0; k < w; k++) exc = Op::op(exc, shw[k]);
  }
  int acc = Op::op(prefix, exc);
#pragma unroll
  for (int k = 0; k < kScanItems; k++) {
    const int nv = Op::op(acc, vals[k]);
    sh[threadIdx.x * kScanItems + k] = acc;
    acc = nv;
  }
  if (kPrefix && total_dev && threadIdx.x == 0 && blockIdx.x == gridDim.x - 1)
    *total_dev = Op::op(prefix, total);
  __syncthreads();
#pragma unroll
  for (int k = 0; k < kScanItems; k++) {
    const int i = base + k * kScanThreads + threadIdx.x;
    if (i < n) out[i] = sh[k * kScanThreads + threadIdx.x];
  }
}

__global__ void k_fill_int(int *p, int value, int n) {
  for (int i = blockIdx.x * blockDim.x + threadIdx.x; i < n; i += gridDim.x * blockDim.x)
    p[i] = value;
}

template <class Op>
void scan_impl(Ctx &c, const int *in, int *out, int n, int *total_dev) {
  if (n <= 0) {
    if (total_dev) fill_int(c, total_dev, 0, 1);
    return;
  }
  const int nb = (n + kScanTile - 1) / kScanTile;
  if (nb > c.scan_blk_cap) {
    if (c.scan_blk) (void)hipFree(c.scan_blk);
    c.scan_blk_cap = nb + 1024;
    if (hipMalloc(&c.scan_blk, sizeof(int) * c.scan_blk_cap) != hipSuccess) {
      c.scan_blk = nullptr;
      c.scan_blk_cap = 0;
      c.err = "scan scratch allocation failed";
      return;
    }
  }
  hipLaunchKernelGGL((k_scan_reduce<Op>), dim3(nb), dim3(kScanThreads), 0, c.stream, in, n,
                     c.scan_blk);
  if (nb <= kScanFusedTiles) {
    hipLaunchKernelGGL((k_scan_down<Op, true>), dim3(nb), dim3(kScanThreads), 0,
                       c.stream, in, n, c.scan_blk, out, total_dev);
    return;
  }
  hipLaunchKernelGGL((k_scan_blocks<Op>), dim3(1), dim3(kScanThreads), 0, c.stream, c.scan_blk,
                     nb, total_dev);
  hipLaunchKernelGGL((k_scan_down<Op, false>), dim3(nb), dim3(kScanThreads), 0,
                     c.stream, in, n, c.scan_blk, out, nullptr);
}

// ---- small sorts -------------------------------------------------------------
// Up to kSmallTiles tiles of 4096 pairs take two launches instead of 32: each tile
// is sorted in LDS by one block, then every pair finds its place: its place in its own
// tile plus, for every other tile, the number of pairs that go before it, by binary
// searches that do not depend on each other.  Ties go to the earlier tile, so the sort
// is stable.
//
// What moves in a tile's passes is a word of 8 bytes, the leading 52 bits of the key
// and the pair's place in the input; keys and values stay where they were loaded.
// Passes over the leading 40 bits (32 in smaller tiles) tell almost all keys of a tile
// apart.  The pairs that agree in them find their places among each other; if more
// than kTileRun do, the tile is sorted by every digit, from the order that it has: that
// costs less than looking through longer runs (half of 2^16 particles on one point: 60 us
// with 8, 76 with 32, 226 with 256; Plummer, clustered and disk systems: the same 33).
//
// Bound by latency and, on the few CUs that have a tile, by the ranking's vector
// instructions; the merge by the number of its loads.  Small tiles are cheaper (1024
// pairs 7.6 us, 2048 12, 4096 20), the searches grow with the square of their number
// (8 tiles 6 us, 16 tiles 11).  So 1024 pairs up to 8 tiles, 2048 up to 16, and 4096.
// Sort and merge at 2^10, 10^4, 3*10^4 and 2^16 pairs: 8, 18, 22 and 31 us; with eight
// passes in tiles of 4096, keys and values moving, 28, 36, 36 and 41; in passes of
// three launches 117 at 2^10 and 163 at 2^16.  Searches 16 at a time spill; with three
// probes for two steps the merge at 2^16 took 13 us.
constexpr int kTileThreads = 1024;
constexpr int kTileWaves = kTileThreads / kWave;
constexpr int kTileRounds = kSortTile / kTileThreads;
constexpr int kSmallTiles = 32;
constexpr int kTileRun = 16;   // the longest run of a tile that is put in order by itself

// keys_out and vals_out may be keys and vals (a single tile is sorted in place): a block
// has its whole tile in LDS before its first store, and reads nothing after that.
template <int ROUNDS>
__global__ __launch_bounds__(kTileThreads) void k_tile_sort(const uint64_t *keys, const int *vals,
                                                            int n, int key_bits,
                                                            uint64_t *keys_out, int *vals_out) {
  BT_BUILD_PRIO();
  static_assert(ROUNDS <= kTileRounds && kSortTile == 4096, "places of 12 bits");
  constexpr int kPairs = ROUNDS * kTileThreads;
  constexpr int kTileLow = ROUNDS == kTileRounds ? 24 : 32;   // bits without a pass
  __shared__ uint64_t skeys[kPairs], swords[kPairs];
  __shared__ int svals[kPairs];
  __shared__ __align__(16) unsigned short wcnt[kTileWaves][256];
  __shared__ __align__(16) int sh_wave[kTileWaves];
  __shared__ int sh_long;
  const int tid = threadIdx.x, lane = lane_id();
  const int w = wave_uniform(tid >> 6);
  const int base = blockIdx.x * kPairs;
  const int tile_n = min(kPairs, n - base);
  if (tid == 0) sh_long = 0;
  // keys have fewer than 64 bits: the pairs past the end, all ones, stay last
  uint64_t ww[ROUNDS];
  int vv[ROUNDS];
#pragma unroll
  for (int r = 0; r < ROUNDS; r++) {   // without branches: all loads in flight together
    const int j = min((w * ROUNDS + r) * kWave + lane, tile_n - 1);
    ww[r] = keys[base + j];
    vv[r] = vals[base + j];
  }
#pragma unroll
  for (int r = 0; r < ROUNDS; r++) {
    const int j = (w * ROUNDS + r) * kWave + lane;
    const uint64_t key = j < tile_n ? ww[r] : ~0ull;
    skeys[j] = key;
    svals[j] = vv[r];
    ww[r] = ((key << (64 - key_bits)) & ~0xFFFull) | (uint64_t)j;
  }
  auto pass = [&](auto digit) {
    reinterpret_cast<uint64_t *>(wcnt[w])[lane] = 0;   // this wave's counters
    wave_lds_sync();
    int dd[ROUNDS], rr[ROUNDS];
#pragma unroll
    for (int r = 0; r < ROUNDS; r++) {
      const int d = digit(ww[r]);
      const uint64_t peers = same_digit(~0ull, d);
      const int rank = lanes_before(peers);
      const int before = wcnt[w][d];
      wave_lds_sync();
      if (rank == 0) wcnt[w][d] = (unsigned short)(before + __popcll(peers));
      wave_lds_sync();
      dd[r] = d;
      rr[r] = before + rank;
    }
    __syncthreads();
    // thread 4d + q: digit d in waves 4q to 4q + 3, the order in which places are given
    int cnt[4], total = 0;
#pragma unroll
    for (int k = 0; k < 4; k++) total += cnt[k] = wcnt[4 * (tid & 3) + k][tid >> 2];
    const int incl = wave_incl_scan(total);
    if (lane == kWave - 1) sh_wave[w] = incl;
    __syncthreads();
    int acc = incl - total;
#pragma unroll
    for (int k = 0; k < kTileWaves; k++) acc += k < w ? sh_wave[k] : 0;
#pragma unroll
    for (int k = 0; k < 4; k++) {
      wcnt[4 * (tid & 3) + k][tid >> 2] = (unsigned short)acc;
      acc += cnt[k];
    }
    __syncthreads();
#pragma unroll
    for (int r = 0; r < ROUNDS; r++) swords[wcnt[w][dd[r]] + rr[r]] = ww[r];
    __syncthreads();
#pragma unroll
    for (int r = 0; r < ROUNDS; r++) ww[r] = swords[(w * ROUNDS + r) * kWave + lane];
  };
#pragma unroll 1
  for (int shift = kTileLow; shift < 64; shift += 8)
    pass([&](uint64_t word) { return (int)(word >> shift) & 0xFF; });
  int place[ROUNDS];
#pragma unroll
  for (int r = 0; r < ROUNDS; r++) {
    const int j = (w * ROUNDS + r) * kWave + lane;
    place[r] = j;
    if ((int)(ww[r] & 0xFFF) >= tile_n) continue;
    const uint64_t key = skeys[ww[r] & 0xFFF];
    int seen = 0;
    for (int k = j - 1; k >= 0; k--) {
      const uint64_t x = swords[k];
      if ((x ^ ww[r]) >> kTileLow) break;
      place[r] -= skeys[x & 0xFFF] > key ? 1 : 0;
      if (++seen >= kTileRun) break;
    }
    for (int k = j + 1; k < tile_n && seen < kTileRun; k++) {
      const uint64_t x = swords[k];
      if ((x ^ ww[r]) >> kTileLow) break;
      place[r] += skeys[x & 0xFFF] < key ? 1 : 0;
      seen++;
    }
    if (seen >= kTileRun) sh_long = 1;
  }
  __syncthreads();
  if (sh_long) {   // by every digit, from this order
#pragma unroll 1
    for (int shift = 0; shift < key_bits; shift += 8)
      pass([&](uint64_t word) { return (int)(skeys[word & 0xFFF] >> shift) & 0xFF; });
#pragma unroll
    for (int r = 0; r < ROUNDS; r++) place[r] = (w * ROUNDS + r) * kWave + lane;
  }
#pragma unroll
  for (int r = 0; r < ROUNDS; r++) {
    const int j = (int)(ww[r] & 0xFFF);
    if (j < tile_n) {
      keys_out[base + place[r]] = skeys[j];
      vals_out[base + place[r]] = svals[j];
    }
  }
}

// One pair per thread; kTileSearches tiles are searched at a time, so that their
// loads are in flight together.
constexpr int kTileSearches = 8;

template <int TILE>
__global__ __launch_bounds__(256) void k_tile_merge(const uint64_t *__restrict__ keys,
                                                    const int *__restrict__ vals, int n,
                                                    uint64_t *__restrict__ keys_out,
                                                    int *__restrict__ vals_out) {
  BT_BUILD_PRIO();
  const int i = blockIdx.x * 256 + threadIdx.x;
  if (i >= n) return;
  const int own = i / TILE;   // uniform over the block
  const int ntiles = (n + TILE - 1) / TILE;
  const uint64_t x = keys[i];
  int place = i - own * TILE;
  for (int t0 = 0; t0 < ntiles; t0 += kTileSearches) {
    int pos[kTileSearches], len[kTileSearches];
    const uint64_t *tile[kTileSearches];
#pragma unroll
    for (int q = 0; q < kTileSearches; q++) {
      const int t = t0 + q;
      tile[q] = keys + (size_t)min(t, ntiles - 1) * TILE;
      len[q] = t < ntiles && t != own ? min(TILE, n - t * TILE) : 0;
      pos[q] = 0;
    }
#pragma unroll
    for (int step = TILE; step >= 1; step >>= 1) {
#pragma unroll
      for (int q = 0; q < kTileSearches; q++) {
        // pairs of earlier tiles go before an equal key, those of later ones after
        const int p = pos[q] + step;
        const uint64_t y = tile[q][max(min(p, len[q]) - 1, 0)];
        const bool before = t0 + q < own ? y <= x : y < x;
        if (p <= len[q] && before) pos[q] = p;
      }
    }
#pragma unroll
    for (int q = 0; q < kTileSearches; q++) place += pos[q];
  }
  keys_out[place] = x;
  vals_out[place] = vals[i];
}

template <int ROUNDS>
void tile_sort_pairs(Ctx &c, uint64_t *keys, int *vals, uint64_t *keys_tmp, int *vals_tmp, int n,
                     int key_bits) {
  constexpr int kPairs = ROUNDS * kTileThreads;
  const int ntiles = (n + kPairs - 1) / kPairs;
  const bool one = ntiles == 1;
  hipLaunchKernelGGL(k_tile_sort<ROUNDS>, dim3(ntiles), dim3(kTileThreads), 0, c.stream, keys,
                     vals, n, key_bits, one ? keys : keys_tmp, one ? vals : vals_tmp);
  if (!one)
    hipLaunchKernelGGL(k_tile_merge<kPairs>, dim3((n + 255) / 256), dim3(256), 0, c.stream,
                       keys_tmp, vals_tmp, n, keys, vals);
}

template <typename T>
void dev_free_raw(T *&p) {
  if (p) (void)hipFree(p);
  p = nullptr;
}

}  // namespace

int grid_for(int n, int block, int cap) {
  int g = (n + block - 1) / block;
  if (g < 1) g = 1;
  if (g > cap) g = cap;
  return g;
}

void fill_int(Ctx &c, int *p, int value, int n) {
  if (n <= 0) return;
  hipLaunchKernelGGL(k_fill_int, dim3(grid_for(n, 256, 4096)), dim3(256), 0, c.stream, p, value,
                     n);
}

void scan_exclusive_sum(Ctx &c, const int *in, int *out, int n, int *total_dev) {
  scan_impl<OpSum>(c, in, out, n, total_dev);
}

// Sorts (keys, vals)[0..n) stably by the low key_bits bits of the key; when
// by_system_after is set, one or two more stable passes order by the system
// of each value (systems of a forest stay contiguous).  The result is left in
// keys/vals; keys_tmp/vals_tmp are scratch of the same size.
//
// short_ok: the passes over the lowest digits may be left out.  40 bits, 13 octal
// digits, tell almost all particles apart, and the gather that follows every sort
// puts the runs of the others in order on its way (place_in_run), reading 8 B per
// pair more instead of 32 B in each of three passes.  5 or 6 passes, so that with
// the systems' the number is odd and the pairs end in keys_tmp.  2*10^7 pairs: the
// passes 1.59 -> 0.97 ms, the PH gather 0.25 -> 0.39 ms, the tree gather as before.
int radix_sort_pairs(Ctx &c, uint64_t *keys, int *vals, uint64_t *keys_tmp, int *vals_tmp,
                     int n, int key_bits, bool by_system_after, bool short_ok) {
  if (n <= 1) return 0;
  const int nblocks = (n + kSortTile - 1) / kSortTile;
  // One system, few tiles, whole keys below the all-ones pad
  if (nblocks <= kSmallTiles && !(by_system_after && c.nsys > 1) && key_bits < 64 &&
      !c.sort_onesweep) {
    if (n <= 8 * kTileThreads)
      tile_sort_pairs<1>(c, keys, vals, keys_tmp, vals_tmp, n, key_bits);
    else if (n <= 16 * 2 * kTileThreads)
      tile_sort_pairs<2>(c, keys, vals, keys_tmp, vals_tmp, n, key_bits);
    else
      tile_sort_pairs<kTileRounds>(c, keys, vals, keys_tmp, vals_tmp, n, key_bits);
    return 0;
  }
  const int hist_n = 256 * nblocks + 256;   // a row per digit, and the digits' totals
  if (hist_n > c.sort_hist_cap) {
    if (c.sort_hist) (void)hipFree(c.sort_hist);
    c.sort_hist_cap = hist_n;
    if (hipMalloc(&c.sort_hist, sizeof(int) * hist_n) != hipSuccess) {
      c.sort_hist = nullptr;
      c.sort_hist_cap = 0;
      c.err = "sort histogram allocation failed";
      return 0;
    }
  }
  struct Pass { int shift, by_sys; };
  std::vector<Pass> passes;
  const int sys_passes = !(by_system_after && c.nsys > 1) ? 0
                         : c.nsys > 65536 ? 3 : c.nsys > 256 ? 2 : 1;
  const int digits = sys_passes & 1 ? 6 : 5;   // of a short sort
  const int low = short_ok && !c.full_sort && !c.sort_onesweep && key_bits > 8 * digits
                      ? key_bits - 8 * digits : 0;
  for (int s = low; s < key_bits; s += 8) passes.push_back({s, 0});
  for (int k = 0; k < sys_passes; k++) passes.push_back({8 * k, 1});
  uint64_t *ks = keys, *kd = keys_tmp;
  int *vs = vals, *vd = vals_tmp;
  if (c.sort_onesweep && (int)passes.size() <= kMaxSortPasses) {
    const int np = (int)passes.size();
    const int ntiles = (n + kOsTile - 1) / kOsTile;
    if (ntiles > c.sort_tiles_cap || !c.sort_hpart) {
      dev_free_raw(c.sort_hpart);
      dev_free_raw(c.sort_gcount);
      dev_free_raw(c.sort_status);
      dev_free_raw(c.sort_ctr);
      c.sort_tiles_cap = 0;
      if (hipMalloc(&c.sort_hpart, sizeof(int) * kSortHistBlocks * kMaxSortPasses * 256) ||
          hipMalloc(&c.sort_gcount, sizeof(int) * kMaxSortPasses * 256) ||
          hipMalloc(&c.sort_status, sizeof(unsigned int) * 2 * 256 * (size_t)ntiles) ||
          hipMalloc(&c.sort_ctr, sizeof(int) * 2)) {
        c.err = "sort scratch allocation failed";
        return 0;
      }
      c.sort_tiles_cap = ntiles;
      hipLaunchKernelGGL(k_sort_clear, dim3(1024), dim3(256), 0, c.stream, c.sort_status,
                         2 * 256 * ntiles, c.sort_ctr);
      hipLaunchKernelGGL(k_sort_clear, dim3(1), dim3(64), 0, c.stream, c.sort_status, 0,
                         c.sort_ctr + 1);
    }
    PassSet ps;
    ps.np = np;
    ps.nsys = c.nsys;
    ps.off = c.d_off;
    for (int k = 0; k < np; k++) {
      ps.shift[k] = passes[k].shift;
      ps.bysys[k] = passes[k].by_sys;
    }
    hipLaunchKernelGGL(k_radix_hist_all, dim3(kSortHistBlocks), dim3(kSortThreads), 0, c.stream,
                       keys, vals, n, ps, c.sort_hpart, c.dc);
    hipLaunchKernelGGL(k_radix_hist_sum, dim3(np, 8), dim3(256), 0, c.stream, c.sort_hpart, np,
                       kSortHistBlocks, c.sort_gcount);
    // pass k uses status buffer k & 1; every sort starts on a clean buffer 0
    const size_t words = (size_t)256 * c.sort_tiles_cap;
    for (int k = 0; k < np; k++) {
      const int cur = k & 1, nxt = cur ^ 1;
      DigitSrc src{passes[k].shift, c.nsys, c.d_off};
      auto kern = passes[k].by_sys ? k_radix_onesweep<true> : k_radix_onesweep<false>;
      hipLaunchKernelGGL(kern, dim3(ntiles), dim3(kSortThreads), 0, c.stream, ks, vs, n, src,
                         c.sort_gcount + 256 * k, c.sort_status + cur * words,
                         c.sort_status + nxt * words, c.sort_ctr + cur, c.sort_ctr + nxt,
                         ntiles, c.dc, kd, vd);
      std::swap(ks, kd);
      std::swap(vs, vd);
    }
    if (np & 1)   // the last pass used buffer 0: clear it for the next sort
      hipLaunchKernelGGL(k_sort_clear, dim3(grid_for(ntiles, 1, 1024)), dim3(256), 0, c.stream,
                         c.sort_status, 256 * ntiles, c.sort_ctr);
  } else {
  for (const Pass &p : passes) {
    DigitSrc src{p.shift, c.nsys, c.d_off};
    auto hist = p.by_sys ? k_radix_hist<true> : k_radix_hist<false>;
    auto scatter = p.by_sys ? k_radix_scatter<true> : k_radix_scatter<false>;
    hipLaunchKernelGGL(hist, dim3(nblocks), dim3(kCThreads), 0, c.stream, ks, vs, n, src,
                       nblocks, c.sort_hist);
    int *total = c.sort_hist + 256 * nblocks;
    hipLaunchKernelGGL(k_radix_rows, dim3(256), dim3(kRowThreads), 0, c.stream, nblocks,
                       c.sort_hist, total);
    hipLaunchKernelGGL(scatter, dim3(nblocks), dim3(kCThreads), 0, c.stream, ks, vs, n, src,
                       nblocks, c.sort_hist, total, kd, vd);
    std::swap(ks, kd);
    std::swap(vs, vd);
  }
  }
  if (low > 0) return low;
  if (ks != keys) {
    (void)hipMemcpyAsync(keys, ks, sizeof(uint64_t) * n, hipMemcpyDeviceToDevice, c.stream);
    (void)hipMemcpyAsync(vals, vs, sizeof(int) * n, hipMemcpyDeviceToDevice, c.stream);
  }
  return 0;
}

}  // namespace bt
