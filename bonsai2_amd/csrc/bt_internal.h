// bt_internal.h -- context state and kernel launchers of libbonsai2_amd.so.
#pragma once
#include <hip/hip_runtime.h>
#include <stdint.h>

#include <string>
#include <vector>

#include "../../include/bonsai2_amd.h"

namespace bt {

constexpr int kSortErr = 8;   // DevCounters::err bit: a sort pass's look-back wait timed out
// DevCounters::err bits: the tree's or the groups' keys held a run of equal leading
// digits too long to be put in order after a short sort (radix_sort_pairs).  The
// phases that follow do nothing; the host sorts again, with every digit, and the
// context keeps to that (Ctx::full_sort).
constexpr int kShortTree = 16, kShortPh = 32;
constexpr int kShortErr = kShortTree | kShortPh;
constexpr int kLevels = 32;   // level table slots (reference int2[32], code/Treecode.h:171)
constexpr int kFp64Levels = 4;     // cells at levels <= this combine moments in FP64

struct MlpDev;   // matrix-core operands of the opening-angle network (bt_learn.h)

// Device buffers of one training-pair collection (bt_learn_collect).
struct LearnBuffers {
  int nsel = 0;
  int *gsel = nullptr;
  float theta_lo = 0.25f, theta_hi = 1.0f;
  int *count = nullptr;
  int max_pairs = 0;
  int2 *pairs = nullptr;
  double *tneed = nullptr;
  double *amag = nullptr;
  float *feat = nullptr, *target = nullptr, *err = nullptr, *tneed_f = nullptr;
  float *sink = nullptr;
};

// Device-resident counters of one context (one allocation).
// Blocks of the walk's statistics reduction (4 words of partials each).
constexpr int kWalkStatBlocks = 256;

// FP32 walks: stack entries per wave kept in LDS (bt_set_walk_lds_stack).
constexpr int kLdsStack = 1024;
#ifndef BT_LDS_STACK_MIN
#define BT_LDS_STACK_MIN 512   // the children one walk step can push (8 * 64)
#endif

struct DevCounters {
  int lvl_start[kLevels + 2];
  int lvl_count[kLevels + 2];
  int lvl_total[kLevels];   // cells per level as counted ([0]: leaves), before the capacity check
  int nnodes, nleaves, nlevels, ncells;
  int ngroups;
  int flags;   // BT_FLAG_*
  int err;     // 1 = cell capacity, 2 = group capacity, 4 = walk stack, 8 = sort,
               // 16, 32 = short sort (kShortTree, kShortPh)
  int queue;   // walk group queue head
  int stack_max;  // deepest walk stack of the last walk (entries)
  int xq[8];      // walk group queues, one per XCD range
  // per-step check of the learned angle, decided on the device
  int fallback;     // 1: the last check failed and the fixed-angle walk ran
  int checks, fallbacks;   // judged so far; checks seeds the sample indices
  // Sticky state, cleared only by the host (launch_clear_sticky) at the start
  // of each API call that steps or walks: every error bit any phase raised
  // since (err is cleared by each phase for itself), the deepest walk stack of
  // every walk since, and the closing half kicks done since.  After an error
  // the kick and drift kernels do nothing, so a failed step leaves the
  // particles as after its first half kick and drift.
  int err_sticky;
  int stack_hw;
  int steps_done;
  // of the last walk: direct_sum, direct_max, approx_sum, approx_max, and 1/2 sum m phi
  unsigned long long wstats[4];
  double wpot;
};

// All threads of one block, of the last kernel that changes the counters before the
// host reads them: the counters to pinned memory (host is null where nothing reads
// them).  A copy after the kernel would be a launch more.
__device__ __forceinline__ void write_counters(const DevCounters *dc, DevCounters *host) {
  if (!host) return;
  static_assert(sizeof(DevCounters) % sizeof(int) == 0, "copied by words");
  const int *src = reinterpret_cast<const int *>(dc);
  int *dst = reinterpret_cast<int *>(host);
  for (int k = threadIdx.x; k < (int)(sizeof(DevCounters) / sizeof(int)); k += blockDim.x)
    __hip_atomic_store(dst + k,
                       __hip_atomic_load(src + k, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT),
                       __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_SYSTEM);
}

// Before every walk: its queues, its stack's depth and its error.
__device__ __forceinline__ void reset_walk(DevCounters *dc) {
  dc->queue = 0;
  dc->stack_max = 0;
  for (int x = 0; x < 8; x++) dc->xq[x] = 0;
  atomicAnd(&dc->err, ~4);
}

__device__ __forceinline__ void clear_sticky(DevCounters *dc) {
  dc->err_sticky = 0;
  dc->stack_hw = 0;
  dc->steps_done = 0;
}

// The values captured graphs bake into their kernel arguments: a graph is
// replayed only while all of them are unchanged (compared bytewise).
struct GraphKey {
  double dt, eps, theta;
  int nleaf, level_split, ncrit;
  int opening, kahan, quadrupole, walk_variant, stack_ints, blocks_per_cu, lds_stack, group_mode;
  int wave_walk;
  int overlap, full_sort;
  float learn_shift, learn_theta_lo, learn_theta_hi;
  int check_ns;
  float check_p99;
  unsigned long long check_seed;
};

struct Ctx {
  int dev = 0;
  // Treecode<double>: particle and cell arrays hold double4 / double2 (twice
  // the float4 / float2 element count is allocated) and the step computes in
  // FP64; otherwise Treecode<float>
  bool fp64 = false;
  hipStream_t stream = nullptr;
  bool own_stream = false;
  double eps = 0.01, theta = 0.75;   // a float context holds float values
  int ncrit = 64, nleaf = 16, level_split = 1;

  // sizes
  int n = 0, cap_n = 0, nsys = 1, max_sys_n = 0;
  std::vector<int> h_off;
  int *d_off = nullptr;

  // particles: "current" arrays hold input order until the first build, then
  // tree order.  *_2 are the reorder targets.
  float4 *pos = nullptr, *vel = nullptr, *pos2 = nullptr, *vel2 = nullptr;
  int *id = nullptr, *id2 = nullptr;

  // sort buffers
  uint64_t *keyB = nullptr;   // sort scratch
  int *valA = nullptr, *valB = nullptr;
  int *sort_hist = nullptr;   // 256 x blocks
  int sort_hist_cap = 0;
  // one-sweep passes: per-pass digit counts of every pass (from one histogram
  // launch), tile status words (two buffers, pass parity) and tile counters
  int *sort_hpart = nullptr;        // kSortHistBlocks x passes x 256 partial counts
  int *sort_gcount = nullptr;       // passes x 256 global digit counts
  unsigned int *sort_status = nullptr;  // 2 x tiles x 256
  int *sort_ctr = nullptr;          // 2 tile counters
  int sort_tiles_cap = 0;
  bool sort_onesweep = false;
  bool full_sort = false;   // sort by every digit (a short sort met too long a run)
  // low key bits the last sort left unsorted (the sorted pairs are then in keyB and
  // valB, and the gather that follows puts them in order)
  int geo_low = 0, ph_low = 0;
  bool ids_in_order = false;   // id[k] = k: no gather since the particles were set
  uint64_t *geo_keys = nullptr;   // sorted geometric keys (tree order)

  // scans
  int *scan_blk = nullptr;
  int scan_blk_cap = 0;

  // boxes
  float4 *box = nullptr;       // per system {cx, cy, cz, hsize}
  float4 *bbox_part = nullptr; // partial min/max
  int bbox_blocks = 1;

  // cells
  int cap_cells = 0;
  uint4 *cells = nullptr;
  float4 *csize = nullptr, *cmono = nullptr, *cq0 = nullptr;
  float2 *cq1 = nullptr, *cls = nullptr;
  float4 *cscr = nullptr;      // 5 float4 per cell (bottom-up moments)
  float4 *cwalk = nullptr;     // 3 float4 per cell: walk record (com,M) -7.5(Qxx,Qyy,Qzz,Qxy) (-7.5Qxz,-7.5Qyz,trQ,1.5trQ)
  uint4 *cell_raw = nullptr;   // the cells in octant order, before [nodes][leaves] of each parent
  int *cell_fin = nullptr, *cell_nch = nullptr;  // their final slots and child counts
  int *cell_arrived = nullptr; // per node: children whose moments are done (0 between launches)
  int *cell_cnt = nullptr;     // cells per level and tile of particles, then their prefixes
  int2 *level_beg = nullptr;   // int2[32] (reference d_level_begIdx)
  int2 *root_cells = nullptr;  // per system (first level-1 cell, count)

  // PH order
  float4 *pos_ph = nullptr;
  int *perm = nullptr;         // PH index -> tree index
  int *id_ph = nullptr;        // PH index -> input index
  uint64_t *ph_keys = nullptr; // sorted PH keys
  float4 *acc = nullptr;       // (ax, ay, az, phi) in PH order

  // groups
  int cap_groups = 0;
  int2 *groups = nullptr;
  int *group_sys = nullptr;
  int *gtmp0 = nullptr, *gtmp1 = nullptr;  // N-sized scan scratch
  int2 *gcounts = nullptr;     // per group (n_approx, n_direct)
  double *gpot = nullptr;      // per group sum m*phi

  // walk
  int *stack = nullptr;
  size_t stack_alloc = 0;
  int stack_ints = 16384;
  int lds_stack = kLdsStack;   // FP32 walks: stack entries per wave kept in LDS
  int group_mode = 0;   // 0: PH-key groups (makeGroups); 1: leaves; 2: tree cells <= ncrit
  int walk_blocks = 0;         // persistent grid (blocks of 256)
  int blocks_per_cu = 0;
  bool wave_walk = false;      // blocks_per_cu set by the caller: one wave per group
  int kahan = 1;
  int walk_variant = 0;        // 0: LDS j-data, 1: scalar loads, 2: two i-particles per lane
  int quadrupole = 1;          // 0: monopole-only P2C (the reference without QUADRUPOLE)
  int num_cus = 256;
  unsigned long long *d_wpart = nullptr;   // partials of the walk's statistics
  // the walk results in hc are those of the last walk queued
  bool wstats_valid = false;

  // learned opening angle
  float2 *sys_scale = nullptr;   // per system (root half size, total mass)
  float *mlp_params = nullptr;   // 1377 FP32 master parameters
  float *mlp_m = nullptr, *mlp_v = nullptr;  // Adam moments
  MlpDev *mlp_dev = nullptr;     // FP16 per-lane operands for inference
  bool have_mlp = false;
  int opening = 0;               // 0 fixed theta, 1 learned per-pair theta
  float learn_shift = 0.f, learn_theta_lo = 0.25f, learn_theta_hi = 1.0f;
  int check_ns = 0;              // FP64 samples re-checked after each learned walk
  float check_p99 = 1e-3f;       // above this p99 the step falls back to fixed theta
  unsigned long long check_seed = 1;
  // 4 * ns ints: the draws' indices into the particle arrays as they were when
  // drawn, the draws' input ids sorted, the draw slot of each sorted id, and
  // each draw's PH index (filled once the step's groups exist)
  int *d_check_idx = nullptr;
  double *d_check = nullptr;     // direct results (4 * ns) + {p50, p99, max}
  // A step sums the check's FP64 forces on stream3 beside the build, from the
  // particles as the drift left them (the tree-order gather writes the other
  // particle buffer).  check_state: 0 no sum queued for the coming check, 1
  // queued on the context stream, 2 queued on stream3 (joins the context
  // stream at chk_join_ev).  check_slices: source slices of the sum (fewer
  // slices leave the build kernels room on the CUs)
  hipStream_t stream3 = nullptr;
  hipEvent_t chk_fork_ev = nullptr, chk_join_ev = nullptr;
  int check_state = 0;
  // Four blocks on every CU: a step of 2^24 (halo + disk, learned) takes 30.9 ms with
  // 512 or 768 slices, whose sum runs into the walk, 29.8 with 1024, 30.3 with 1280 and
  // more, which hold the build back; of 2^22 7.20, 7.02, 6.99 and 7.03 ms.
  int check_slices = 1024;

  // energies / direct sum scratch
  double *d_energy = nullptr;  // 2 * nsys
  double *d_direct = nullptr;
  int direct_cap = 0;

  DevCounters *dc = nullptr;
  DevCounters *pinned_dc = nullptr;   // where read_counters or a kernel copies them
  DevCounters hc;                     // as last read

  // moveParticles' half kick still owed: the next computeForces closes the
  // kick-drift-kick step with it (0 = none)
  double pending_kick = 0.0;
  int check_cap = 0;             // samples d_check / d_check_idx are sized for

  // state
  bool have_particles = false, have_tree = false, have_mp = false, have_groups = false,
       have_acc = false;

  // captured step (bt_step_graph).  The tree-order gather writes the particles
  // into the other of two buffers, so there is one graph per buffer holding
  // the particles at the start of the step: [0] for graph_pos0, [1] for the other.
  hipGraph_t graph[2] = {nullptr, nullptr};
  hipGraphExec_t graph_exec[2] = {nullptr, nullptr};
  float4 *graph_pos0 = nullptr;
  GraphKey graph_key{};   // every by-value launch parameter the graphs hold
  int tree_version = 0;

  // timing
  hipEvent_t ev[12] = {};
  // A step runs the groups (PH keys, PH sort, groups) on stream2 beside the
  // level build and multipoles on stream: both need only the tree-order
  // particles and sorted keys (overlap = false runs them in sequence on
  // stream).  forked: the last step's phase events follow that layout
  // (multipoles end at ev[10], groups at ev[11]).
  hipStream_t stream2 = nullptr;
  hipEvent_t fork_ev = nullptr, join_ev = nullptr;
  bool overlap = true;
  bool forked = false;
  float ms[10] = {};
  bool timing = true;

  std::string err;
};

// ---- launchers (each queues work on c.stream) --------------------------
void launch_bbox(Ctx &c);
void launch_geo_keys(Ctx &c);
void launch_gather_tree(Ctx &c);
// read: the last kernel writes the counters to c.pinned_dc (also below)
void launch_levels(Ctx &c, bool read = false);
int max_cell_tiles(int n);   // c.cell_cnt holds kCellCntRows ints per tile
constexpr int kCellCntRows = 22;
void launch_multipoles(Ctx &c);

// Sorts (keys, vals) by the low key_bits bits, or, if short_ok, possibly by fewer of
// the leading ones: returns the number of low bits left unsorted, the pairs then in
// keys_tmp and vals_tmp (0: sorted, in keys and vals).
int radix_sort_pairs(Ctx &c, uint64_t *keys, int *vals, uint64_t *keys_tmp, int *vals_tmp,
                     int n, int key_bits, bool by_system_after, bool short_ok);
void scan_exclusive_sum(Ctx &c, const int *in, int *out, int n, int *total_dev);
void fill_int(Ctx &c, int *p, int value, int n);

void launch_ph_keys(Ctx &c);
// the PH gather of the particles and the groups
void launch_groups(Ctx &c, bool read = false);
// groups = tree cells (mode 1: the leaves; mode 2: cells of <= ncrit
// particles), in tree order; the group order is the tree order
void launch_leaf_groups(Ctx &c);

// run_if: device flag; the walk (reset, traversal, statistics) does nothing
// unless it is nonzero (nullptr = always run)
void launch_walk(Ctx &c, const int *run_if = nullptr, bool clear = false, bool read = false,
                 bool reset = true);
bool walk_stats_in_one(const Ctx &c);   // the walks that can do so
bool walk_as_team(const Ctx &c);        // the four waves of a block walk a group together
// Stack entries no walk can exceed: a step pops 64 cells and pushes at most 512,
// so at most 448 more than it takes stay behind on each of the 21 levels.  A
// context whose stack may be too small keeps to one wave per group, so that the
// same calls report BT_ERR_STACK.
constexpr int kSafeStack = 8 + 21 * 448;

void launch_mlp_prepare(Ctx &c);
void launch_mlp_forward(Ctx &c, int n, const float *x, float *y);
void launch_sys_scale(Ctx &c);
void launch_learn_pairs(Ctx &c, LearnBuffers &L);
void launch_learn_errors(Ctx &c, LearnBuffers &L, int npairs);
void launch_learn_amag(Ctx &c, int ns, const int *d_idx, const double *d_direct, double *amag);
int mlp_grad_blocks();
void launch_mlp_grad(Ctx &c, const float *params, int n, const float *feat, const float *target,
                     int batch, unsigned long long seed, int step, float *partial);
// the rows of partial summed: grad[kMlpParams] and the loss behind it, or an Adam
// update with them and the loss alone
void launch_mlp_reduce(Ctx &c, const float *partial, int batch, double *grad);
void launch_mlp_adam(Ctx &c, float *p, float *m, float *v, const float *partial, int batch,
                     double *loss, float lr, int step);
// targets of the next check, drawn on the device from check_seed and the
// device's check count: indices into the current particle arrays (c.pos,
// c.id), and their input ids sorted for launch_check_map
void launch_check_idx(Ctx &c, int ns);
// each target's PH index (after the step's groups), from c.id_ph
void launch_check_map(Ctx &c, int ns);
// p50/p99/max of the relative force errors into out[0..2]; sets the device's
// fallback flag (p99 > check_p99) and counts checks and fallbacks
void launch_learn_check(Ctx &c, int ns, const int *d_idx, const double *d_direct, double *out);

// closing: the second half kick of a step (counted in steps_done)
void launch_kick(Ctx &c, double dt_half, bool closing = false, bool read = false);
// the opening half kick (dth) and the drift (dt) of a step, in one pass
void launch_kick_drift(Ctx &c, double dth, double dt, bool clear);   // resets the walk too
void launch_clear_sticky(Ctx &c);
hipError_t launch_iota(Ctx &c, int n, int *out);   // out[k] = k
// n values of the context's 4-vector type: dst[idx[k]] = src[k] (scatter) or
// dst[k] = src[idx[k]]
hipError_t launch_permute(Ctx &c, bool scatter, const int *idx, const void *src, void *dst);
void launch_energies(Ctx &c);
int direct_slices(int ns);   // d_out of launch_direct: ns * (slices + 1) double4
void launch_direct(Ctx &c, int ns, const int *d_idx, double *d_out, bool check = false);
// src: the particles targets and sources are read from (null: c.pos_ph)
void launch_direct_parts(Ctx &c, int ns, const int *d_idx, double *d_out, double *d_part,
                         int slices, bool check = false, const void *src = nullptr);

// host-side helpers
int grid_for(int n, int block, int cap);

}  // namespace bt
