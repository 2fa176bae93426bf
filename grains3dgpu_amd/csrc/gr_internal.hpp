// gr_internal.hpp -- device data layout and launchers shared by the kernel
// translation units (gr_broad.hip, gr_narrow64.hip, gr_narrow32.hip) and
// the C-ABI (gr_capi.hip).
//
// HBM layout (N particles, E candidate entries, C cells):
//   state    pos[3][N], quat[4][N] (x,y,z,w), vel[3][N], omega[3][N]   FP64 planes
//   ids      shape[N], sim[N]                                          u32
//   broad    key[N] (by particle: the reference's cell, each step),
//            skey[N] (the search's cell), key/idx ping-pong [2][N], rank[N],
//            cell_off[C+1] (first sorted position of each search cell) u32
//   sorted   bp[N] = {x, y, z, list radius}   32 B, cell order, as the lists
//            were built; rcs[N] = prefilter radius
//            bp32[N] = bp in FP32, relative to the sim's domain minimum, 16 B
//            cell_sph[C] = bounding sphere of each cell's residents, 16 B
//            pk[N] = PoseRec {pos, quat, shape, sim}  64 B, vk[N] = VelRec
//            {vel, omega}  48 B, cell order (gathered from the planes when
//            the lists are built; the steps advance these, and the planes
//            are written by a run's last step and before the next build:
//            neighbours of a cell are contiguous, so the gathers of a wave
//            share cache lines)
//   pairs    cand[K][N] (k-major: lanes write consecutive words),
//            cand_count[N], entry_off[N+1]                            u32
//            pair_i[E], pair_j[E] (sorted positions), pair_flag[E]     u32
//            pair_res[E] = {F[3], M[3]} in the narrow-phase type (FP64
//            for FP32-mixed with GRAINS_FP64_CONTACTS: its contacts are
//            all FP64 re-runs)
//   shapes   ShapeNP<double>[S], ShapeNP<float>[S], ShapeDyn[S]
#pragma once

#include <hip/hip_runtime.h>
#include <stdint.h>

#include "gr_geom.hpp"

namespace gr {

constexpr int kBlock = 256;          // threads per block of streaming kernels
constexpr int kItems = 8;            // items per thread in sort / scan tiles
constexpr int kTile = kBlock * kItems;
constexpr int kRadixMaxBits = 11;    // widest radix digit (LDS histograms of 2048 counters)
constexpr int kRadixMaxDigits = 1 << kRadixMaxBits;
constexpr double kPrefilterSlack = 1.e-10;
constexpr int kMaxMovers = 4096;     // particles that change cell in a step, merged into the previous order
constexpr uint32_t kSmallSort = 8192; // the most particles k_sort_small can hold (64 KB of LDS)
constexpr uint32_t kSmallSortDefault = 1024;  // beds up to this size sort in one block by default
// beds up to this size integrate every particle with its walls in one launch:
// touching superquadrics, one launch and two, us: 2,000 30 and 49, 8,000 27 and
// 51, 16,000 31 and 51, 20,000 36 and 51, 30,000 51 and 52, 45,000 58 and 54
// (larger beds also integrate beside the searches; spheres by 32,000: 52 and
// 60 us a step)
constexpr uint64_t kWideIntegrate = 16384;
constexpr uint32_t kXcds = 8;          // dies of the card, each with its own L2; blocks go to them in turn
constexpr int kMaxNarrowPerCu = 64;  // resident narrow-phase blocks per CU the queue buffers are sized for

// Velocities of the particle at one sorted position.
struct alignas(16) VelRec {
  double v[3], w[3];
};

// per-pair flag bits
constexpr uint32_t kFlagContact = 1u;
constexpr uint32_t kFlagGjk = 2u;
constexpr uint32_t kFlagDeep = 4u;
constexpr uint32_t kFlagRefine = 8u;
constexpr uint32_t kFlagCand = 16u;     // passed the bounding-sphere prefilter this step
constexpr int kFlagSlot = 8;            // contacts: the neighbour cell's slot in the visit order, from this bit on

// device counters (u64), summed over the steps of one grains_step call.
// Each counter is spread over kCntSlots words (slot = block index mod
// kCntSlots, summed on the host): one word would serialise an atomic per
// wave at a single L2 channel (~12 ns each, 190 us for 1e6 particles).
constexpr int kCntSlots = 128;
enum Counter {
  kCntCandidates = 0,
  kCntGjk,
  kCntGjkIters,
  kCntContacts,
  kCntWall,
  kCntOod,
  kCntDeep,
  kCntRefine,
  kCntOverflow,
  kCntMaxCand,   // stored as max
  kCntBackup,
  kCntDeferred,  // entries the screening pass queued
  kCntMaxIters,  // stored as max: the longest GJK search
  kCntNear,      // FP32-mixed: decisions within the rounding band (re-run in FP64)
  kCntNan,       // particle-steps whose new state is not finite
  kCntRefIters,  // FP32-mixed: GJK iterations of the FP64 re-runs
  kCntRefMaxIters,  // stored as max: the longest FP64 re-run
  kNumCounters = 18
};

// State of the neighbour lists and of the run of steps (device words, read
// back with the counters).
enum ListState {
  kNlValid = 0,   // the lists cover the current positions (2: for one step only)
  kNlRun,         // this step runs (latched from kNlValid by its first kernel)
  kNlLast,        // it is the run's last step, or a checkpoint's
  kNlDone,        // steps of the run taken
  kNlTarget,      // steps of the run asked for (recorded: up to the next checkpoint)
  kNlOver,        // a list outgrew max_neighbors when the lists were built; 2: with its skin, 3: kNlOutside with
                  // a skin -- no step uses such lists
  kNlOutside,     // a centre lay outside a periodic side when they were built
  kNlStale,       // the records by sorted position are ahead of the state's planes
  kNlWords = 8
};

// One simulation's linked cell and forces.
struct SimGrid {
  double lo[3], hi[3], L[3];
  double h;
  double g[3];
  uint32_t n3[3];
  uint32_t base;         // first global cell
  int32_t periodic;      // bitmask x=1, y=2, z=4
  uint32_t table;        // first entry of its contact table block
  uint32_t obs_begin, obs_end;  // its obstacles (obstacles sorted by sim)
  double half_skin;      // half the lists' skin: added to every list radius
  double move2;          // squared displacement since the lists were built up to which they hold
};

// What an FP64 search found of a contact: the closest points of the cores in
// their own frames, their distance, and whether they overlap.
struct alignas(64) GjkRec {
  double pa[3], pb[3], dist, deep;
};

// Where the steps of a recorded trajectory leave their states (device memory,
// set before each chunk of steps): 13 planes per slot, step number kNlDone of
// the run in slot first + kNlDone, slots [1, slots).
struct StateLog {
  double* base;
  int64_t first;
  uint64_t slots;
};

// Dynamics of one shape (RigidBody mass properties, RigidBody.cpp:19-59);
// inertia and its inverse as upper triangles xx xy xz yy yz zz.
struct Dynamics {
  double mass;
  double inertia[6], inv[6];
};
// As the device stores it: one 64-byte line for the shapes whose principal
// axes are their own (all but general polyhedra), a second for the rest.
struct alignas(64) ShapeDyn {
  double mass;
  double diag[3], inv_diag[3];
  double off_axis;  // 1: the second line holds products of inertia
  double off[3], inv_off[3], pad[2];
};

// Exponents and axis ratios of a superquadric's crust core as the FP64
// support chain divides them out (sq_support_pow), once per shape.
struct alignas(64) SqPow {
  double k1, k2, g, r, in1;  // 1/(n2-1), 1/(n1-1), (n1-n2)/(n2 (n1-1)), n1/n2, 1/n1
  double ba, ca, cb;         // b/a, c/a, c/b
};

template <class T>
struct alignas(16) PairRes {
  T f[3];
  T m[3];
};

// Pose of the particle at one sorted position: one 64-byte line.
struct alignas(64) PoseRec {
  double x, y, z;
  double qx, qy, qz, qw;
  uint32_t shape, sim;
};

struct DevScene {
  uint64_t n;
  uint32_t nsims, nobs, nmat;
  // state (planes of length n)
  double *pos, *quat, *vel, *omega;
  uint32_t *shape, *sim;
  // shapes
  const ShapeNP<double>* np64;
  const ShapeNP<float>* np32;
  const SqPow* sq64;
  const ShapeDyn* dyn;
  const double* rc_pf;          // prefilter radius per shape
  const double* verts64;        // full polyhedron vertices
  const double* cverts64;       // crust-core vertices
  const float* verts32;
  const float* cverts32;
  const HookeP<double>* hooke64;
  const HookeP<float>* hooke32;
  const SimGrid* grids;         // the reference's cells (keys, adjacency, visit order)
  const SimGrid* sgrids;        // the search's cells (with a skin at least a list reach wide, else the reference's)
  const uint32_t* obs_shape;    // sorted by sim
  const double* obs_tr;         // 12 doubles each
  // broad phase
  uint32_t *key, *skey, *keyA, *idxA, *keyB, *idxB, *rank;
  uint32_t* rkey;               // reference cell by sorted position when the lists were built
  double* rcs;                  // prefilter radius by sorted position
  uint32_t* nl;                 // ListState words
  int32_t skin;                 // 1: the lists hold for several steps; 0: for the step they are built in
  int32_t keep_torce;           // 1: every step's total force and torque are stored (the adjoint reads them)
  const uint32_t* sidx;         // particle at each sorted position (this step)
  uint32_t* cell_off;           // CSR over cells: residents of c are [off[c], off[c+1])
  double4* bp;                  // {x, y, z, list radius} by sorted position when the lists were built
  float4* bp32;                 // bp in FP32, positions relative to the sim's domain minimum
  float4* cell_sph;             // per cell: bounding sphere of its residents' spheres (bp32 frame)
  PoseRec* pk;                  // pose by sorted position
  VelRec* vk;                   // velocities by sorted position
  double* hk;                   // integration history by sorted position (12 values each; d.ab_hist)
  double* rws;                  // largest radius by sorted position (with obstacles)
  uint32_t ncells;
  uint32_t *hist;               // 256 * n_tiles (+1)
  uint32_t *scan_blocks;        // block sums of scans
  // pairs
  uint32_t K;
  uint64_t ecap;
  uint32_t *cand, *cand_count, *entry_off;
  uint32_t *pair_i, *pair_j, *pair_flag;
  void* pair_res;               // PairRes<T>[ecap]
  StateLog* log;                // recorded trajectories
  GjkRec* gjk_rec;              // by entry: the contacts' searches (reverse sweep of the adjoint; else null)
  uint32_t* refine_list;        // entries to re-run in FP64 (FP32-mixed)
  uint32_t* refine_count;
  uint32_t* queue_next;         // FP64 searches: entries handed out past the dealt ones
  uint32_t* defer_list;         // entries the screening pass left undecided: kDeferQueues
                                // queues of defer_cap words, block b filling queue b % kDeferQueues
  uint32_t* defer_count;        // their lengths (one 64-byte line each)
  uint32_t defer_cap;
  int32_t split;                // 1: screening pass + pass over the queued entries
  int32_t cand_staged;          // 1: candidate search stages neighbour windows in LDS
  int32_t cand_half;            // 1 (direct search): each unordered pair tested once, lists sorted by k_expand
  int32_t half_wl;              // 1: the half-shell search takes its groups from a work list (dense cells)
  uint32_t* half_goff;          // work list: groups per cell, scanned (ncells + 1)
  uint32_t* half_glist;         // work list: each group's cell (n)
  int32_t balls;                // 1: every particle is a sphere
  int32_t gen_obs;              // 1: some obstacle is not a Rectangle (GJK in the integration kernel)
  // time integration: scheme, and its history (12 planes of n): for
  // ADAMS_BASHFORTH the previous step's v, w, a, alpha (NaN: none yet), for
  // LEAPFROG plane 0 NaN until the first (half) kick
  int32_t integrator;
  double* ab_hist;
  // GRAINS_WARM_START (FP32-mixed, physics semantics): each entry's GJK
  // direction of its last step, in the world frame, in two buffers of K x N
  // records {x, y, z, neighbour id as bits} in entry order, and per particle
  // id the first entry and the entry count (ws_nb); ws_par = the buffer of
  // the current lists (flipped when they are built: the other holds the
  // records of the lists before, k_warm_carry)
  int32_t warm;
  float4* ws;
  uint2* ws_nb;
  uint32_t* ws_par;
  // particles (sorted positions) within reach of an obstacle, queued by k_integrate for
  // k_integrate_obs (count reset by the step's first kernel)
  uint32_t* obs_list;
  uint32_t* obs_count;
  // the particles k_integrate_pend queues for k_integrate_obs (steps with
  // the integration beside the narrow phase: the settled particles' queue
  // is integrated on the second stream, this one after the join); count
  // obs_count + 2
  uint32_t* obs_list2;
  uint32_t* obs_count2;
  // Two narrow passes: pend[s] = 1 when the screen left an entry of sorted
  // position s undecided (both particles of the entry are marked; cleared by
  // the integration).  On large beds the integration of the other particles runs
  // while the complete pass and the FP64 re-runs settle those entries, and
  // the marked particles (queued in pend_list, count pend_count, reset by
  // the screen) are integrated after both.
  // Sorting by merge.  sort_state[0] = 1 once a sorted order and its
  // inverse permutation stand (k_cells; cleared when the state is set),
  // [2] = the particles that changed search cell (k_hash; at most kMaxMovers of
  // their ids kept in mv_list); the step's sort follows from the two
  // (sort_mode: 0 radix, 1 merge the movers into the previous order, 2 no
  // particle changed cell), evaluated by each sort kernel itself.  The
  // merge's movers sorted by (key << 32 | id) (mv_keys), their previous
  // positions sorted (mv_old), their new positions (mv_dst).
  uint32_t* sort_state;
  int32_t small_sort;           // 1: k_sort_small sorts the bed (n <= GRAINS_SMALL_SORT_MAX, default 1,024)
  uint32_t* mv_list;
  uint64_t* mv_keys;
  uint32_t* mv_old;
  uint32_t* mv_dst;
  uint32_t* pend;
  uint32_t* pend_list;
  uint32_t* pend_count;
  // per particle outputs
  int32_t* contact_count;
  double *last_force, *last_torque;
  unsigned long long* counters;
  // launch shape of the per-particle / per-entry kernels
  uint32_t block;               // threads per block (64, 128, 256)
  uint32_t narrow_blocks;       // blocks of the persistent narrow-phase launch
  // config
  double dt;
  uint32_t flags;
  double gjk_rel;
  double gjk_rel64;             // FP32-mixed: GJK tolerance of the FP64 re-runs
  int32_t res64;                // FP32-mixed with FP64 contact geometry: pair_res holds PairRes<double>
  int precision;
};

// Buffers of one backward step of the adjoint sweep (gr_adjoint.hip).
struct AdjBufs {
  double* state;          // 13 planes (pos 3, quat 4, vel 3, omega 3): the state at step t
  double* abar;           // 13 planes: in, the adjoint of the state at t+1; out, at t
  double* own;            // 13 planes: a particle's own partial (integration, walls)
  double *Fb, *Mb;        // 3 planes each: adjoint of the total force and torque
  double *part_i, *part_j;  // 13 per entry: the entry's partials for its two particles
  double* entry_theta;    // 4 per entry: kn, en, etat, muc
  uint32_t* entry_tidx;   // contact-table entry of each entry (~0: none)
  double* wall_theta;     // 4 per (particle, wall slot)
  uint32_t* wall_tidx;
  uint32_t max_obs;       // wall slots per particle
  GjkRec* gjk;            // d.gjk_rec during the sweep, or null: k_adj_entry searches again
  double* dtheta;         // 4 per contact-table entry, summed over the sweep
};

// ---- launchers ------------------------------------------------------------------
// gr_broad.hip
void launch_fill_u32(uint32_t* p, uint64_t n, uint32_t v, hipStream_t s);
// keys_prev: the sort's output buffer (the previous step's sorted keys)
void launch_sq_pow(const ShapeNP<double>* np, SqPow* out, uint64_t n, hipStream_t s);
void launch_store_state(const DevScene& d, hipStream_t s);
void launch_log_state(const DevScene& d, hipStream_t s);
void launch_log_set(const DevScene& d, StateLog v, uint32_t target, hipStream_t s);
void launch_state_rows(const DevScene& d, uint64_t i0, uint64_t m, double* out, hipStream_t s);
void launch_hash(const DevScene& d, const uint32_t* keys_prev, hipStream_t s);
// sorts (d.key, identity) into the returned buffers: `passes` LSD passes of
// `digit_bits` (8 .. kRadixMaxBits) bits each
void launch_sort(DevScene& d, int passes, int digit_bits, uint32_t** keys_sorted, uint32_t** idx_sorted,
                 hipStream_t s);
// cell ranges, inverse permutation and the sorted pose records
// the step's pairs by particle: off[n + 1] (off[n] their number), nb their neighbours
struct PairLists {
  const uint32_t *off, *nb;
};
PairLists launch_pair_lists(const DevScene& d, uint32_t want, bool list, hipStream_t s);
const uint32_t* launch_key_order(const DevScene& d, int passes, int digit_bits, hipStream_t s);
void launch_cells(const DevScene& d, const uint32_t* keys_s, const uint32_t* idx_s, hipStream_t s);
void launch_candidates(const DevScene& d, const uint32_t* keys_s, hipStream_t s);
// exclusive scan of min(in[i], clamp) into out[0 .. n]; gate (optional):
// the kernels return at once unless *gate == 0
void launch_scan(const uint32_t* in, uint32_t* out, uint64_t n, uint32_t* block_sums, hipStream_t s,
                 uint32_t clamp = 0xffffffffu, const uint32_t* gate = nullptr);
// the start of a run of n steps: counters cleared, run words set; fresh: the
// lists and the sorted order no longer stand, the planes hold the state
void launch_run_begin(const DevScene& d, uint32_t n, bool fresh, hipStream_t s);
void launch_expand(const DevScene& d, hipStream_t s);
int cu_count();
// gr_narrow64.hip / gr_narrow32.hip
// pass 0: every entry (complete, or screened with d.split);
// pass 1: the entries the screen queued (no launch unless d.split)
void launch_narrow64(const DevScene& d, int pass, hipStream_t s);
void launch_narrow32(const DevScene& d, int pass, hipStream_t s);
void launch_refine64(const DevScene& d, hipStream_t s);
// part 0: every particle; 1: the particles the screen did not mark (the
// marked ones queued); 2: the queued ones.  Each part then integrates the
// particles it queued near obstacles, except part 1 (part 2 does it).
void launch_integrate64(const DevScene& d, hipStream_t s, int part = 0);
void launch_integrate32(const DevScene& d, hipStream_t s, int part = 0);
// gr_adjoint.hip: one backward step (the forward step t must have just run)
void launch_adjoint_step(const DevScene& d, const AdjBufs& a, uint32_t n_tables, hipStream_t s);
// standalone GJK distance batches (GrainsTestDev workload)
// shapes in host memory, at most kArgShapes and no polyhedra
constexpr int kArgShapes = 8;
void launch_gjk_batch_args64(const ShapeNP<double>* shapes, size_t count, const uint32_t* sa, const uint32_t* sb,
                             const double* ta, const double* tb, uint64_t n, GjkArgs args, double* dist,
                             int32_t* iters, hipStream_t s);
void launch_gjk_batch_args32(const ShapeNP<float>* shapes, size_t count, const uint32_t* sa, const uint32_t* sb,
                             const double* ta, const double* tb, uint64_t n, GjkArgs args, double* dist,
                             int32_t* iters, hipStream_t s);
void launch_gjk_batch64(const ShapeNP<double>* shapes, const double* verts, const uint32_t* sa,
                        const uint32_t* sb, const double* ta, const double* tb, uint64_t n,
                        GjkArgs args, double* dist, double* pa, double* pb, int32_t* iters,
                        hipStream_t s);
void launch_gjk_batch32(const ShapeNP<float>* shapes, const float* verts, const uint32_t* sa,
                        const uint32_t* sb, const double* ta, const double* tb, uint64_t n,
                        GjkArgs args, double* dist, double* pa, double* pb, int32_t* iters,
                        hipStream_t s);

// ---- small device helpers --------------------------------------------------------
// The screening pass's queues: one counter would serialise a block's append
// at a single address (~12 ns each).
constexpr uint32_t kDeferQueues = 16;
__device__ __forceinline__ uint32_t defer_total(const DevScene& d) {
  uint32_t t = 0;
#pragma unroll
  for (uint32_t q = 0; q < kDeferQueues; ++q) t += d.defer_count[16 * q];
  return t;
}
// the k-th queued entry, the queues end to end
__device__ __forceinline__ uint32_t defer_entry(const DevScene& d, uint32_t k) {
  uint32_t q = 0;
#pragma unroll
  for (uint32_t i = 0; i + 1 < kDeferQueues; ++i) {
    const uint32_t c = d.defer_count[16 * i];
    if (q == i && k >= c) {
      k -= c;
      q = i + 1;
    }
  }
  return d.defer_list[(uint64_t)q * d.defer_cap + k];
}
// The reference's cell of a centre (LinkedCell::computeLinearCellHash,
// LinkedCell.cpp:117-149), FP64 divide + floor; the partial last cell beyond
// n3 h (the domain is rarely a multiple of h) folds into cell n3 - 1, and
// centres outside (a NaN: cell 0) into the border cells.
__device__ __forceinline__ void cell_of(const SimGrid& g, const double* p, uint32_t* c) {
#pragma unroll
  for (int k = 0; k < 3; ++k) {
    const double f = floor((p[k] - g.lo[k]) / g.h);
    if (!(f >= 0.0))
      c[k] = 0;
    else if (f >= (double)g.n3[k])
      c[k] = g.n3[k] - 1;
    else
      c[k] = (uint32_t)f;
  }
}
__device__ __forceinline__ uint32_t cell_key(const SimGrid& g, const uint32_t* c) {
  return g.base + (c[2] * g.n3[1] + c[1]) * g.n3[0] + c[0];
}
// Slot of cell cj among the 27 neighbour cells of ci in the visit order (z
// outer, then y, then x: LinkedCell.cpp:41-70), periodic axes wrapped; -1:
// not a neighbour.
__device__ __forceinline__ int cell_slot(const SimGrid& g, const uint32_t* ci, const uint32_t* cj) {
  int dd[3];
#pragma unroll
  for (int k = 0; k < 3; ++k) {
    const int n = (int)g.n3[k];
    int v = (int)cj[k] - (int)ci[k];
    if ((g.periodic >> k) & 1) v = v == n - 1 ? -1 : (v == 1 - n ? 1 : v);
    if (v < -1 || v > 1) return -1;
    dd[k] = v;
  }
  return ((dd[2] + 1) * 3 + dd[1] + 1) * 3 + dd[0] + 1;
}
// The step's sort from sort_state (DevScene::sort_state): radix when no
// previous order stands or too many particles changed cell, a merge when a
// few did, nothing when none did.  Read between k_hash and k_cells, which
// write the two words, so every sort kernel of a step sees the same mode.
__device__ __forceinline__ uint32_t sort_mode(const uint32_t* st) {
  const uint32_t moved = st[2];
  return !st[0] ? 0u : (moved == 0 ? 2u : (moved <= (uint32_t)kMaxMovers ? 1u : 0u));
}
__device__ __forceinline__ uint32_t wave_sum(uint32_t v) {
#pragma unroll
  for (int o = 32; o > 0; o >>= 1) v += __shfl_xor(v, o);
  return v;
}
__device__ __forceinline__ uint32_t wave_max(uint32_t v) {
#pragma unroll
  for (int o = 32; o > 0; o >>= 1) v = max(v, (uint32_t)__shfl_xor(v, o));
  return v;
}
// add a per-lane count to device counter `which`, one atomic per wave on
// the block's slot
__device__ __forceinline__ void count_add(unsigned long long* counters, int which, uint32_t v) {
  uint32_t s = wave_sum(v);
  if (__lane_id() == 0 && s)
    atomicAdd(&counters[which * kCntSlots + (blockIdx.x & (kCntSlots - 1))], (unsigned long long)s);
}
__device__ __forceinline__ void count_max(unsigned long long* counters, int which, uint32_t v) {
  uint32_t m = wave_max(v);
  if (__lane_id() == 0 && m)
    atomicMax(&counters[which * kCntSlots + (blockIdx.x & (kCntSlots - 1))], (unsigned long long)m);
}
// append `val` of every lane with `pred` to list[*count ...] in block-local
// (LDS) `count`, one LDS atomic per wave; called by all active lanes
__device__ __forceinline__ void block_append(uint32_t* list, uint32_t* count, bool pred, uint32_t val) {
  const unsigned long long mask = __ballot(pred);
  if (!mask) return;
  const int leader = __ffsll(mask) - 1;
  const uint32_t lane = __lane_id();
  uint32_t base = 0;
  if ((int)lane == leader) base = atomicAdd(count, (uint32_t)__popcll(mask));
  base = __shfl(base, leader);
  if (pred) list[base + (uint32_t)__popcll(mask & ((1ull << lane) - 1ull))] = val;
}
// append `val` of every lane with `pred` to list[*count ...], one atomic per
// wave (lanes keep their order within the wave); called by all active lanes
__device__ __forceinline__ void wave_append(uint32_t* list, uint32_t* count, bool pred, uint32_t val) {
  const unsigned long long mask = __ballot(pred);
  if (!mask) return;
  const int leader = __ffsll(mask) - 1;
  const uint32_t lane = __lane_id();
  uint32_t base = 0;
  if ((int)lane == leader) base = atomicAdd(count, (uint32_t)__popcll(mask));
  base = __shfl(base, leader);
  if (pred) list[base + (uint32_t)__popcll(mask & ((1ull << lane) - 1ull))] = val;
}

// Quaternion state and pose helpers
__device__ __forceinline__ Qt<double> load_quat(const double* q, uint64_t n, uint64_t i) {
  return {q[i], q[n + i], q[2 * n + i], q[3 * n + i]};
}
__device__ __forceinline__ V3<double> load3(const double* p, uint64_t n, uint64_t i) {
  return {p[i], p[n + i], p[2 * n + i]};
}
__device__ __forceinline__ void store3(double* p, uint64_t n, uint64_t i, V3<double> v) {
  p[i] = v.x;
  p[n + i] = v.y;
  p[2 * n + i] = v.z;
}
// particle i's state into the planes, from its records at sorted position s
__device__ __forceinline__ void store_state(const DevScene& d, uint64_t i, uint64_t s, const PoseRec& p,
                                            const VelRec& v) {
  const uint64_t n = d.n;
  store3(d.pos, n, i, {p.x, p.y, p.z});
  d.quat[i] = p.qx;
  d.quat[n + i] = p.qy;
  d.quat[2 * n + i] = p.qz;
  d.quat[3 * n + i] = p.qw;
  store3(d.vel, n, i, {v.v[0], v.v[1], v.v[2]});
  store3(d.omega, n, i, {v.w[0], v.w[1], v.w[2]});
  if (d.hk)
    for (int k = 0; k < 12; ++k) d.ab_hist[k * n + i] = d.hk[12 * s + k];
}
__device__ __forceinline__ Dynamics load_dyn(const ShapeDyn* p) {
  const double4* q = (const double4*)p;  // the first line at once
  const double4 a = q[0], b = q[1];
  Dynamics r = {a.x, {a.y, 0.0, 0.0, a.z, 0.0, a.w}, {b.x, 0.0, 0.0, b.y, 0.0, b.z}};
  if (b.w != 0.0) {
    r.inertia[1] = p->off[0], r.inertia[2] = p->off[1], r.inertia[4] = p->off[2];
    r.inv[1] = p->inv_off[0], r.inv[2] = p->inv_off[1], r.inv[4] = p->inv_off[2];
  }
  return r;
}
// minimum-image offset along periodic directions
__device__ __forceinline__ V3<double> min_image(const SimGrid& g, V3<double> d) {
  if (g.periodic & 1) d.x -= g.L[0] * rint(d.x / g.L[0]);
  if (g.periodic & 2) d.y -= g.L[1] * rint(d.y / g.L[1]);
  if (g.periodic & 4) d.z -= g.L[2] * rint(d.z / g.L[2]);
  return d;
}
// ContactForceModelBuilderFactory::computeHash (ContactForceModelBuilderFactory.cpp:77-83)
__device__ __forceinline__ uint32_t material_hash(uint32_t x, uint32_t y) {
  uint32_t s = x < y ? x : y, l = x < y ? y : x;
  return l * (l + 1) / 2 + s;
}

}  // namespace gr
