// gr_broad.hip -- linked-cell broad phase on the device: the neighbour lists'
// build (spheres grown by half the lists' skin), the state's planes and rows.
//
//   k_hash        cell key of every particle (LinkedCell::computeLinearCellHash,
//                 LinkedCell.cpp:117-149), FP64 divide + floor as the reference
//   radix sort    stable LSD sort of (key, index), digits of 8-11 bits (the
//                 fewest passes for the key width): per-tile LDS
//                 histogram, device-wide exclusive scan, stable scatter ranked
//                 with wave ballots (replaces thrust::sort_by_key,
//                 ComponentManagerGPU.cpp:282-285)
//   k_cells       CSR cell offsets from the sorted keys (the cell start/end of
//                 ComponentManagerGPU_Kernels.cpp:28-75), the inverse
//                 permutation and the pose records in cell order
//   k_candidates_half / _half_wl
//                 per cell, each unordered pair tested once
//   k_candidates_direct / _staged
//                 per particle, the 27 cells in the reference order
//                 (LinkedCell.cpp:41-70) and their residents ascending
//                 (ComponentManagerCPU.cpp:364-421), bounding-sphere prefilter;
//                 the second stages the block's neighbour windows in LDS
//   scan/expand   CSR offsets and the flat (i, j) entry list, in sorted
//                 positions
#include <type_traits>
#include <algorithm>

#include "gr_internal.hpp"

namespace gr {

__global__ void k_fill_u32(uint32_t* __restrict__ p, uint64_t n, uint32_t v) {
  uint64_t i = (uint64_t)blockIdx.x * blockDim.x + threadIdx.x;
  if (i < n) p[i] = v;
}

void launch_fill_u32(uint32_t* p, uint64_t n, uint32_t v, hipStream_t s) {
  if (!n) return;
  hipLaunchKernelGGL(k_fill_u32, dim3((unsigned)((n + kBlock - 1) / kBlock)), dim3(kBlock), 0, s, p, n, v);
}

// ---- shapes -----------------------------------------------------------------------
// (FP64 division rounds here as on the host; 10^6 shapes' records were 64 MB
// of divisions and a copy of a new layout)
__global__ void __launch_bounds__(kBlock) k_sq_pow(const ShapeNP<double>* __restrict__ np, SqPow* __restrict__ out,
                                                   uint64_t n) {
  const uint64_t i = (uint64_t)blockIdx.x * blockDim.x + threadIdx.x;
  if (i >= n) return;
  SqPow r = {};
  if (np[i].kind == GRAINS_SUPERQUADRIC) {
    const double a = np[i].core[0], b = np[i].core[1], c = np[i].core[2], n1 = np[i].core[3], n2 = np[i].core[4];
    r = {1.0 / (n2 - 1.0), 1.0 / (n1 - 1.0), (n1 - n2) / (n2 * (n1 - 1.0)), n1 / n2, 1.0 / n1,
         b / a,            c / a,            c / b};
  }
  out[i] = r;
}
void launch_sq_pow(const ShapeNP<double>* np, SqPow* out, uint64_t n, hipStream_t s) {
  hipLaunchKernelGGL(k_sq_pow, dim3((unsigned)((n + kBlock - 1) / kBlock)), dim3(kBlock), 0, s, np, out, n);
}

// ---- the start of a run -------------------------------------------------------------
// fresh: the lists do not stand (nor the sorted order), and the planes hold
// the state, whatever a run that stopped early left in the records.
__global__ void k_run_begin(DevScene d, uint32_t n, int fresh) {
  const uint32_t i = blockIdx.x * blockDim.x + threadIdx.x;
  if (i < (uint32_t)kNumCounters * kCntSlots) d.counters[i] = 0ull;
  if (i == 0) {
    d.nl[kNlDone] = 0u;
    d.nl[kNlTarget] = n;
    if (fresh) d.sort_state[0] = d.sort_state[2] = d.nl[kNlStale] = 0u;
  }
}
void launch_run_begin(const DevScene& d, uint32_t n, bool fresh, hipStream_t s) {
  constexpr unsigned words = kNumCounters * kCntSlots;
  hipLaunchKernelGGL(k_run_begin, dim3((words + kBlock - 1) / kBlock), dim3(kBlock), 0, s, d, n, fresh ? 1 : 0);
}

// ---- cell hash --------------------------------------------------------------------
// The first kernel of a list build (no other kernel runs beside it on the
// stream): ws_par (warm starts on), the warm-start buffer of the lists, is
// flipped here, unless the build before was of no use (kNlOver >= 2): the
// records carried over to its lists are left, and the ones before it carried
// over again.  Keys are those of the search's cells (d.sgrids).
// With a sorted order of the previous build in place (sort_state[0]), a
// particle whose key differs from its key there (ks_prev at its previous
// position rank[i]) has changed cell: it is counted in sort_state[2] and the
// first kMaxMovers are listed in mv_list.
// The steps since the last build have advanced the records by sorted position
// only (kNlStale): the planes take them here.
__global__ void k_hash(DevScene d, const uint32_t* __restrict__ ks_prev) {
  const uint64_t n = d.n;
  uint64_t i = (uint64_t)blockIdx.x * blockDim.x + threadIdx.x;
  bool mover = false;
  if (i == 0) {
    if (d.warm && d.nl[kNlOver] < 2u) d.ws_par[0] = 1u - d.ws_par[0];
    d.nl[kNlValid] = 0u;
    d.nl[kNlOver] = 0u;
    d.nl[kNlOutside] = 0u;
  }
  if (i < n) {
    const SimGrid& g = d.sgrids[d.sim[i]];
    double p[3];
    if (d.nl[kNlStale]) {
      const uint32_t r = d.rank[i];
      const PoseRec q = d.pk[r];
      store_state(d, i, r, q, d.vk[r]);
      p[0] = q.x, p[1] = q.y, p[2] = q.z;
    } else {
      p[0] = d.pos[i], p[1] = d.pos[n + i], p[2] = d.pos[2 * n + i];
    }
    uint32_t c[3];
    cell_of(g, p, c);
    const uint32_t k = cell_key(g, c);
    d.skey[i] = k;
    if (d.sort_state[0]) mover = k != ks_prev[d.rank[i]];
  }
  const unsigned long long mb = __ballot(mover);
  if (mb) {
    const int leader = __ffsll(mb) - 1;
    uint32_t base = 0;
    if ((int)__lane_id() == leader) base = atomicAdd(&d.sort_state[2], (uint32_t)__popcll(mb));
    base = __shfl(base, leader) + (uint32_t)__popcll(mb & ((1ull << __lane_id()) - 1ull));
    if (mover && base < (uint32_t)kMaxMovers) d.mv_list[base] = (uint32_t)i;
  }
}

void launch_hash(const DevScene& d, const uint32_t* keys_prev, hipStream_t s) {
  hipLaunchKernelGGL(k_hash, dim3((unsigned)((d.n + kBlock - 1) / kBlock)), dim3(kBlock), 0, s, d, keys_prev);
}

// the planes of the state a run has reached between two of its steps
__global__ void k_store_state(DevScene d) {
  if (!d.nl[kNlStale]) return;
  const uint64_t i = (uint64_t)blockIdx.x * blockDim.x + threadIdx.x;
  if (i >= d.n) return;
  const uint32_t r = d.rank[i];
  store_state(d, i, r, d.pk[r], d.vk[r]);
}
void launch_store_state(const DevScene& d, hipStream_t s) {
  hipLaunchKernelGGL(k_store_state, dim3((unsigned)((d.n + kBlock - 1) / kBlock)), dim3(kBlock), 0, s, d);
}

// the state after the step just taken, into its slot of the log
__global__ void k_log_state(DevScene d) {
  if (!d.nl[kNlRun] || !d.log->base) return;
  const int64_t slot = d.log->first + (int64_t)d.nl[kNlDone];
  if (slot < 1 || slot >= (int64_t)d.log->slots) return;
  const uint64_t s = (uint64_t)blockIdx.x * blockDim.x + threadIdx.x, n = d.n;
  if (s >= n) return;
  const uint32_t i = d.sidx[s];
  const PoseRec p = d.pk[s];
  const VelRec v = d.vk[s];
  double* o = d.log->base + 13 * n * (uint64_t)slot + i;
  o[0] = p.x, o[n] = p.y, o[2 * n] = p.z;
  o[3 * n] = p.qx, o[4 * n] = p.qy, o[5 * n] = p.qz, o[6 * n] = p.qw;
#pragma unroll
  for (int k = 0; k < 3; ++k) {
    o[(7 + k) * n] = v.v[k];
    o[(10 + k) * n] = v.w[k];
  }
}
void launch_log_state(const DevScene& d, hipStream_t s) {
  hipLaunchKernelGGL(k_log_state, dim3((unsigned)((d.n + kBlock - 1) / kBlock)), dim3(kBlock), 0, s, d);
}
__global__ void k_log_set(DevScene d, StateLog v, uint32_t target) {
  *d.log = v;
  d.nl[kNlTarget] = target;
}
void launch_log_set(const DevScene& d, StateLog v, uint32_t target, hipStream_t s) {
  hipLaunchKernelGGL(k_log_set, dim3(1), dim3(1), 0, s, d, v, target);
}

// Particles [i0, i0 + m) of the state's planes as rows, into the host's
// pinned memory: out = pos[m][3], quat[m][4], vel[m][3], omega[m][3].
__global__ void k_state_rows(DevScene d, uint64_t i0, uint64_t m, double* __restrict__ out) {
  const uint64_t t = (uint64_t)blockIdx.x * blockDim.x + threadIdx.x;
  if (t >= 13 * m) return;
  const double* src = t < 3 * m ? d.pos : t < 7 * m ? d.quat : t < 10 * m ? d.vel : d.omega;
  const uint64_t base = t < 3 * m ? 0 : t < 7 * m ? 3 * m : t < 10 * m ? 7 * m : 10 * m;
  const uint32_t comps = base == 3 * m ? 4u : 3u, r = (uint32_t)(t - base);  // (13 m < 2^32: kRowsMax)
  out[t] = src[(uint64_t)(r % comps) * d.n + i0 + r / comps];
}
void launch_state_rows(const DevScene& d, uint64_t i0, uint64_t m, double* out, hipStream_t s) {
  hipLaunchKernelGGL(k_state_rows, dim3((unsigned)((13 * m + kBlock - 1) / kBlock)), dim3(kBlock), 0, s, d, i0, m, out);
}

// ---- block-wide exclusive scan of one value per thread ---------------------------
__device__ __forceinline__ uint32_t block_exclusive_scan(uint32_t v, uint32_t* lds_waves, uint32_t& total) {
  const int lane = __lane_id();
  const int wave = threadIdx.x / 64;
  uint32_t x = v;
#pragma unroll
  for (int o = 1; o < 64; o <<= 1) {
    uint32_t y = __shfl_up(x, o);
    if (lane >= o) x += y;
  }
  if (lane == 63) lds_waves[wave] = x;
  __syncthreads();
  uint32_t off = 0, tot = 0;
  const int nw = blockDim.x / 64;
  for (int w = 0; w < nw; ++w) {
    uint32_t t = lds_waves[w];
    if (w < wave) off += t;
    tot += t;
  }
  __syncthreads();
  total = tot;
  return off + x - v;
}

// ---- radix sort -----------------------------------------------------------------
// Elements of tile b are b*kTile + k*kBlock + tid, k = 0..kItems-1: the item
// slot k outermost, so a stable rank follows (k, wave, lane).
// BITS-bit digits (8 .. kRadixMaxBits): D = 2^BITS counters per tile, each
// thread owns digits tid, tid + kBlock, ...; hist is digit-major,
// hist[d * ntiles + tile], so one exclusive scan gives every (digit, tile)
// its first output position.
template <int BITS>
__global__ void __launch_bounds__(kBlock) k_radix_hist(uint64_t n, const uint32_t* __restrict__ keys,
                                                      int shift, uint32_t ntiles, uint32_t* __restrict__ hist,
                                                      const uint32_t* __restrict__ gate) {
  if (sort_mode(gate) != 0u) return;  // the step's sort is not the radix sort
  constexpr uint32_t D = 1u << BITS;
  __shared__ uint32_t cnt[D];
  const uint32_t tid = threadIdx.x;
  for (uint32_t dg = tid; dg < D; dg += kBlock) cnt[dg] = 0;
  __syncthreads();
  const uint64_t base = (uint64_t)blockIdx.x * kTile;
#pragma unroll
  for (int k = 0; k < kItems; ++k) {
    uint64_t e = base + (uint64_t)k * kBlock + tid;
    if (e < n) atomicAdd(&cnt[(keys[e] >> shift) & (D - 1u)], 1u);
  }
  __syncthreads();
  for (uint32_t dg = tid; dg < D; dg += kBlock) hist[(uint64_t)dg * ntiles + blockIdx.x] = cnt[dg];
}

template <int BITS>
__global__ void __launch_bounds__(kBlock) k_radix_scatter(uint64_t n, const uint32_t* __restrict__ kin,
                                                         const uint32_t* __restrict__ iin, int shift,
                                                         uint32_t ntiles, const uint32_t* __restrict__ offs,
                                                         uint32_t* __restrict__ kout, uint32_t* __restrict__ iout,
                                                         int identity_in, const uint32_t* __restrict__ gate) {
  if (sort_mode(gate) != 0u) return;  // the step's sort is not the radix sort
  constexpr uint32_t D = 1u << BITS;
  __shared__ uint32_t run[D];
  __shared__ uint32_t wcnt[kBlock / 64][D];
  const uint32_t tid = threadIdx.x;
  const int lane = __lane_id();
  const int wave = tid / 64;
  for (uint32_t dg = tid; dg < D; dg += kBlock) {
    run[dg] = offs[(uint64_t)dg * ntiles + blockIdx.x];
#pragma unroll
    for (int w = 0; w < kBlock / 64; ++w) wcnt[w][dg] = 0;
  }
  __syncthreads();
  const uint64_t base = (uint64_t)blockIdx.x * kTile;
  const uint64_t lt = lane ? (~0ull >> (64 - lane)) : 0ull;
  // the tile's keys and indices are loaded up front: the barriers of the
  // item loop would otherwise wait on one load latency per item
  uint32_t keys[kItems], idxs[kItems];
#pragma unroll
  for (int k = 0; k < kItems; ++k) {
    const uint64_t e = base + (uint64_t)k * kBlock + tid;
    keys[k] = e < n ? kin[e] : 0u;
    idxs[k] = e < n ? (identity_in ? (uint32_t)e : iin[e]) : 0u;
  }
#pragma unroll
  for (int k = 0; k < kItems; ++k) {
    const uint64_t e = base + (uint64_t)k * kBlock + tid;
    const bool valid = e < n;
    const uint32_t key = keys[k];
    const uint32_t idx = idxs[k];
    uint32_t dig = (key >> shift) & (D - 1u);
    // lanes of this wave holding the same digit
    uint64_t m = __ballot(valid);
#pragma unroll
    for (int b = 0; b < BITS; ++b) {
      uint64_t bb = __ballot((dig >> b) & 1u);
      m &= ((dig >> b) & 1u) ? bb : ~bb;
    }
    const uint32_t rank = __popcll(m & lt);
    if (valid && rank == 0) wcnt[wave][dig] = __popcll(m);
    __syncthreads();
    // per digit: offsets of the waves in order, then advance the running count
    for (uint32_t dg = tid; dg < D; dg += kBlock) {
      uint32_t r = run[dg];
#pragma unroll
      for (int w = 0; w < kBlock / 64; ++w) {
        uint32_t c = wcnt[w][dg];
        wcnt[w][dg] = r;
        r += c;
      }
      run[dg] = r;
    }
    __syncthreads();
    if (valid) {
      uint32_t p = wcnt[wave][dig] + rank;
      kout[p] = key;
      iout[p] = idx;
    }
    __syncthreads();
    for (uint32_t dg = tid; dg < D; dg += kBlock) {
#pragma unroll
      for (int w = 0; w < kBlock / 64; ++w) wcnt[w][dg] = 0;
    }
    __syncthreads();
  }
}

// ---- device-wide exclusive scan (block sums, down-sweep) --------------------------
// Values are read as min(in[i], clamp).
__global__ void __launch_bounds__(kBlock) k_scan_reduce(uint64_t n, const uint32_t* __restrict__ in,
                                                       uint32_t* __restrict__ bsum, uint32_t clamp,
                                                       const uint32_t* __restrict__ gate) {
  if (gate && sort_mode(gate) != 0u) return;
  __shared__ uint32_t lw[kBlock / 64];
  const uint64_t base = (uint64_t)blockIdx.x * kTile + (uint64_t)threadIdx.x * kItems;
  uint32_t s = 0;
#pragma unroll
  for (int k = 0; k < kItems; ++k)
    if (base + k < n) s += min(in[base + k], clamp);
  uint32_t tot;
  block_exclusive_scan(s, lw, tot);
  if (threadIdx.x == 0) bsum[blockIdx.x] = tot;
}

// Down-sweep: each block first sums the preceding blocks' sums itself (a few
// hundred at most: cheaper than a separate launch scanning them), then scans
// its tile.  In place (out == in) is safe: a block reads its tile before it
// writes it, and only the block sums are read across blocks.
__global__ void __launch_bounds__(kBlock) k_scan_down(uint64_t n, const uint32_t* __restrict__ in,
                                                     uint32_t* __restrict__ out,
                                                     const uint32_t* __restrict__ bsum, uint32_t nb,
                                                     uint32_t clamp, const uint32_t* __restrict__ gate) {
  if (gate && sort_mode(gate) != 0u) return;
  __shared__ uint32_t lw[kBlock / 64];
  __shared__ uint32_t pw[kBlock / 64];
  uint32_t p = 0;
  for (uint32_t i = threadIdx.x; i < blockIdx.x; i += kBlock) p += bsum[i];
#pragma unroll
  for (int o = 32; o > 0; o >>= 1) p += __shfl_xor(p, o);
  if (__lane_id() == 0) pw[threadIdx.x / 64] = p;
  const uint64_t base = (uint64_t)blockIdx.x * kTile + (uint64_t)threadIdx.x * kItems;
  uint32_t v[kItems];
  uint32_t s = 0;
#pragma unroll
  for (int k = 0; k < kItems; ++k) {
    v[k] = base + k < n ? min(in[base + k], clamp) : 0u;
    s += v[k];
  }
  uint32_t tot;
  uint32_t ex = block_exclusive_scan(s, lw, tot);  // its barriers also publish pw
  uint32_t prefix = 0;
#pragma unroll
  for (int w = 0; w < kBlock / 64; ++w) prefix += pw[w];
  ex += prefix;
#pragma unroll
  for (int k = 0; k < kItems; ++k) {
    if (base + k < n) out[base + k] = ex;
    ex += v[k];
  }
  if (blockIdx.x == nb - 1 && threadIdx.x == 0) out[n] = prefix + tot;
}

// out has n+1 entries; block_sums needs ceil(n/kTile) entries.  One tile: one
// launch.
void launch_scan(const uint32_t* in, uint32_t* out, uint64_t n, uint32_t* block_sums, hipStream_t s,
                 uint32_t clamp, const uint32_t* gate) {
  uint32_t nb = (uint32_t)((n + kTile - 1) / kTile);
  if (nb == 0) nb = 1;
  if (nb > 1) hipLaunchKernelGGL(k_scan_reduce, dim3(nb), dim3(kBlock), 0, s, n, in, block_sums, clamp, gate);
  hipLaunchKernelGGL(k_scan_down, dim3(nb), dim3(kBlock), 0, s, n, in, out, block_sums, nb, clamp, gate);
}

template <int BITS>
static void run_sort_passes(DevScene& d, int passes, const uint32_t*& kin, const uint32_t*& iin, hipStream_t s) {
  const uint64_t n = d.n;
  const uint32_t nt = (uint32_t)((n + kTile - 1) / kTile);
  uint32_t* ko[2] = {d.keyA, d.keyB};
  uint32_t* io[2] = {d.idxA, d.idxB};
  const uint32_t* gate = d.sort_state;  // the radix sort runs in mode 0
  for (int p = 0; p < passes; ++p) {
    const int shift = BITS * p;
    hipLaunchKernelGGL(k_radix_hist<BITS>, dim3(nt), dim3(kBlock), 0, s, n, kin, shift, nt, d.hist, gate);
    launch_scan(d.hist, d.hist, (uint64_t)(1u << BITS) * nt, d.scan_blocks, s, 0xffffffffu, gate);
    hipLaunchKernelGGL(k_radix_scatter<BITS>, dim3(nt), dim3(kBlock), 0, s, n, kin, iin, shift, nt, d.hist,
                       ko[p & 1], io[p & 1], p == 0 ? 1 : 0, gate);
    kin = ko[p & 1];
    iin = io[p & 1];
  }
}

// ---- merging the particles that changed cell -------------------------------------
// The previous order (ks, is) is sorted by (key, id).  Its particles whose
// key did not change keep their keys and their relative order; the movers
// (at most kMaxMovers) are sorted by (new key, id) here and each is placed
// after the stayers below it: the stayers of its new key's previous cell
// range with a lower id, and all before that range, less the movers that
// stood there.  One block; the movers' old positions sorted beside.
__global__ void __launch_bounds__(1024) k_merge_movers(DevScene d, const uint32_t* __restrict__ is) {
  if (sort_mode(d.sort_state) != 1u) return;
  __shared__ uint64_t km[kMaxMovers];
  __shared__ uint32_t om[kMaxMovers];
  const uint32_t cnt = d.sort_state[2];  // <= kMaxMovers in this mode
  const uint32_t t = threadIdx.x;
  // the sort spans the next power of two at or above the count (a bed
  // moves a few particles a step: a few stages instead of 55)
  uint32_t P = 2;
  while (P < cnt) P <<= 1;
  for (uint32_t m = t; m < P; m += blockDim.x) {
    if (m < cnt) {
      const uint32_t i = d.mv_list[m];
      km[m] = ((uint64_t)d.skey[i] << 32) | i;
      om[m] = d.rank[i];
    } else {
      km[m] = ~0ull;
      om[m] = ~0u;
    }
  }
  __syncthreads();
  // bitonic sorts of both arrays, ascending
  for (uint32_t size = 2; size <= P; size <<= 1)
    for (uint32_t stride = size >> 1; stride > 0; stride >>= 1) {
      for (uint32_t m = t; m < P; m += blockDim.x) {
        const uint32_t o = m ^ stride;
        if (o > m) {
          const bool up = (m & size) == 0;
          if ((km[m] > km[o]) == up) {
            const uint64_t x = km[m];
            km[m] = km[o];
            km[o] = x;
          }
          if ((om[m] > om[o]) == up) {
            const uint32_t x = om[m];
            om[m] = om[o];
            om[o] = x;
          }
        }
      }
      __syncthreads();
    }
  for (uint32_t m = t; m < cnt; m += blockDim.x) {
    const uint32_t key = (uint32_t)(km[m] >> 32), id = (uint32_t)km[m];
    // first position of the previous order at or above (key, id): in the
    // previous range of the key, the first id above (a mover is not there:
    // its previous key was another)
    uint32_t lo = d.cell_off[key], hi = d.cell_off[key + 1];
    while (lo < hi) {
      const uint32_t mid = (lo + hi) >> 1;
      if (is[mid] < id)
        lo = mid + 1;
      else
        hi = mid;
    }
    // movers that stood before it
    uint32_t a = 0, b = cnt;
    while (a < b) {
      const uint32_t mid = (a + b) >> 1;
      if (om[mid] < lo)
        a = mid + 1;
      else
        b = mid;
    }
    d.mv_keys[m] = km[m];
    d.mv_dst[m] = lo - a + m;
  }
  for (uint32_t m = t; m < cnt; m += blockDim.x) d.mv_old[m] = om[m];
}

// One thread per previous position s: a stayer moves down by the movers that
// stood before it and up by the movers that now sort before it; a mover is
// placed by k_merge_place.  Into (ko, io).
__global__ void __launch_bounds__(kBlock) k_merge_stayers(DevScene d, const uint32_t* __restrict__ ks,
                                                         const uint32_t* __restrict__ is, uint32_t* __restrict__ ko,
                                                         uint32_t* __restrict__ io) {
  if (sort_mode(d.sort_state) != 1u) return;
  const uint64_t s = (uint64_t)blockIdx.x * blockDim.x + threadIdx.x;
  if (s >= d.n) return;
  const uint32_t i = is[s], k = ks[s];
  if (d.skey[i] != k) return;
  const uint32_t cnt = d.sort_state[2];
  const uint64_t me = ((uint64_t)k << 32) | i;
  uint32_t a = 0, b = cnt;
  while (a < b) {
    const uint32_t mid = (a + b) >> 1;
    if (d.mv_old[mid] < (uint32_t)s)
      a = mid + 1;
    else
      b = mid;
  }
  uint32_t c = 0, e = cnt;
  while (c < e) {
    const uint32_t mid = (c + e) >> 1;
    if (d.mv_keys[mid] < me)
      c = mid + 1;
    else
      e = mid;
  }
  const uint32_t dst = (uint32_t)s - a + c;
  ko[dst] = k;
  io[dst] = i;
}

__global__ void __launch_bounds__(kBlock) k_merge_place(DevScene d, uint32_t* __restrict__ ko,
                                                       uint32_t* __restrict__ io) {
  if (sort_mode(d.sort_state) != 1u) return;
  const uint32_t m = blockIdx.x * blockDim.x + threadIdx.x;
  if (m >= d.sort_state[2]) return;
  const uint64_t km = d.mv_keys[m];
  ko[d.mv_dst[m]] = (uint32_t)(km >> 32);
  io[d.mv_dst[m]] = (uint32_t)km;
}

// the merged order back into the sort's output buffers
__global__ void __launch_bounds__(kBlock) k_merge_copy(DevScene d, const uint32_t* __restrict__ ko,
                                                      const uint32_t* __restrict__ io, uint32_t* __restrict__ ks,
                                                      uint32_t* __restrict__ is) {
  if (sort_mode(d.sort_state) != 1u) return;
  const uint64_t s = (uint64_t)blockIdx.x * blockDim.x + threadIdx.x;
  if (s >= d.n) return;
  ks[s] = ko[s];
  is[s] = io[s];
}

// ---- one-block sort of a small bed -----------------------------------------------
// A bed of at most kSmallSort particles (d.small_sort): its (key, index)
// pairs sorted ascending in one block by a bitonic network in LDS over the
// next power of two -- the stable radix sort's order exactly -- in one launch
// instead of the radix passes and the merge (small beds are bound by their
// launches, not their work).
__global__ void __launch_bounds__(1024) k_sort_small(DevScene d, uint32_t* __restrict__ ko,
                                                     uint32_t* __restrict__ io) {
  __shared__ uint64_t km[kSmallSort];
  const uint32_t n = (uint32_t)d.n, t = threadIdx.x;
  uint32_t P = 2;
  while (P < n) P <<= 1;
  for (uint32_t m = t; m < P; m += blockDim.x) km[m] = m < n ? ((uint64_t)d.skey[m] << 32) | m : ~0ull;
  __syncthreads();
  for (uint32_t size = 2; size <= P; size <<= 1)
    for (uint32_t stride = size >> 1; stride > 0; stride >>= 1) {
      for (uint32_t m = t; m < P; m += blockDim.x) {
        const uint32_t o = m ^ stride;
        if (o > m) {
          const bool up = (m & size) == 0;
          const uint64_t a = km[m], b = km[o];
          if ((a > b) == up) {
            km[m] = b;
            km[o] = a;
          }
        }
      }
      __syncthreads();
    }
  for (uint32_t m = t; m < n; m += blockDim.x) {
    ko[m] = (uint32_t)(km[m] >> 32);
    io[m] = (uint32_t)km[m];
  }
}

static void radix_passes(DevScene& d, int passes, int digit_bits, const uint32_t*& kin, const uint32_t*& iin,
                         hipStream_t s) {
  switch (digit_bits) {
    case 8: run_sort_passes<8>(d, passes, kin, iin, s); break;
    case 9: run_sort_passes<9>(d, passes, kin, iin, s); break;
    case 10: run_sort_passes<10>(d, passes, kin, iin, s); break;
    default: run_sort_passes<11>(d, passes, kin, iin, s); break;
  }
}

void launch_sort(DevScene& d, int passes, int digit_bits, uint32_t** keys_sorted, uint32_t** idx_sorted,
                 hipStream_t s) {
  if (d.small_sort) {
    hipLaunchKernelGGL(k_sort_small, dim3(1), dim3(1024), 0, s, d, d.keyA, d.idxA);
    *keys_sorted = d.keyA;
    *idx_sorted = d.idxA;
    return;
  }
  const uint32_t* kin = d.skey;
  const uint32_t* iin = nullptr;
  radix_passes(d, passes, digit_bits, kin, iin, s);
  uint32_t* ks = const_cast<uint32_t*>(kin);
  uint32_t* is = const_cast<uint32_t*>(iin);
  // the merge (mode 1) works in the other buffer pair
  uint32_t* ko = ks == d.keyA ? d.keyB : d.keyA;
  uint32_t* io = is == d.idxA ? d.idxB : d.idxA;
  const dim3 grid((unsigned)((d.n + kBlock - 1) / kBlock));
  hipLaunchKernelGGL(k_merge_movers, dim3(1), dim3(1024), 0, s, d, is);
  hipLaunchKernelGGL(k_merge_stayers, grid, dim3(kBlock), 0, s, d, ks, is, ko, io);
  hipLaunchKernelGGL(k_merge_place, dim3((kMaxMovers + kBlock - 1) / kBlock), dim3(kBlock), 0, s, d, ko, io);
  hipLaunchKernelGGL(k_merge_copy, grid, dim3(kBlock), 0, s, d, ko, io, ks, is);
  *keys_sorted = ks;
  *idx_sorted = is;
}

// The particles by (key, id) of the reference's cells (d.key), between two
// steps: through the radix passes (or the one block) in arrays that only a step
// or a build fills -- the obstacles', the marked particles' and the candidates'
// -- with a count that is zero then as the sort's state (mode 0).
const uint32_t* launch_key_order(const DevScene& d, int passes, int digit_bits, hipStream_t s) {
  DevScene t = d;
  t.skey = d.key;
  t.keyA = d.obs_list;
  t.idxA = d.obs_list2;
  t.keyB = d.pend_list;
  t.idxB = d.cand;
  t.sort_state = d.refine_count;
  const uint32_t *kin = t.skey, *iin = nullptr;
  if (d.small_sort) {
    hipLaunchKernelGGL(k_sort_small, dim3(1), dim3(1024), 0, s, t, t.keyA, t.idxA);
    return t.idxA;
  }
  radix_passes(t, passes, digit_bits, kin, iin, s);
  return iin;
}

// ---- cell ranges and sorted records -----------------------------------------------
// The CSR offsets of the cells: cell_off[c] = first sorted position whose key
// is >= c (a lower bound in the sorted keys), one thread per offset, so every
// one of the C + 1 offsets is written once, coalesced, and empty cells get
// empty ranges.  (Filling the empty cells from the thread of the particle
// before them serialises the empty layers at the floor and the ceiling of a
// bed on one thread each.)
// The same thread also writes the cell's bounding sphere, cell_sph[c] =
// {centre, R} in the FP32 frame of bp32: every resident's prefilter sphere
// lies inside it (R = max |x_j - centre| + r_j over the residents, inflated
// by 1e-6 of the magnitudes involved, several times the FP32 rounding of
// the records and of this computation); empty cells get R = -inf.  The
// candidate search skips a neighbour cell whose sphere its own cannot reach.
__global__ void k_cell_off(const uint32_t* __restrict__ ks, const float4* __restrict__ bp32, uint64_t n,
                           uint64_t ncells, uint32_t* __restrict__ off, float4* __restrict__ sph) {
  const uint64_t c = (uint64_t)blockIdx.x * blockDim.x + threadIdx.x;
  if (c > ncells) return;
  // lower bound L = min{s : s == n or ks[s] >= c}, galloping from the
  // previous step's offset of the cell (any start in [0, n] gives the same
  // L; cells keep their offsets within a few positions from step to step,
  // so a few dependent loads replace the ~20 of a full binary search)
  auto at_or_after = [&](uint64_t t) { return t >= n || (uint64_t)ks[t] >= c; };
  const uint64_t g = off[c] < n ? off[c] : n;
  uint64_t lo, hi;
  if (!at_or_after(g)) {  // L > g
    lo = g + 1;
    hi = n;
    for (uint64_t step = 1; lo < n; step <<= 1) {
      const uint64_t p = g + step < n ? g + step : n;
      if (at_or_after(p)) {
        hi = p;
        break;
      }
      lo = p + 1;
    }
  } else {  // L <= g
    lo = 0;
    hi = g;
    for (uint64_t step = 1; step <= g; step <<= 1) {
      const uint64_t p = g - step;
      if (!at_or_after(p)) {
        lo = p + 1;
        break;
      }
      hi = p;
    }
  }
  while (lo < hi) {
    const uint64_t mid = (lo + hi) >> 1;
    if (at_or_after(mid))
      hi = mid;
    else
      lo = mid + 1;
  }
  off[c] = (uint32_t)lo;
  if (c == ncells || !sph) return;
  uint64_t end = lo;
  float mn[3] = {3e38f, 3e38f, 3e38f}, mx[3] = {-3e38f, -3e38f, -3e38f};
  while (end < n && (uint64_t)ks[end] == c) {
    const float4 r = bp32[end++];
    mn[0] = fminf(mn[0], r.x), mn[1] = fminf(mn[1], r.y), mn[2] = fminf(mn[2], r.z);
    mx[0] = fmaxf(mx[0], r.x), mx[1] = fmaxf(mx[1], r.y), mx[2] = fmaxf(mx[2], r.z);
  }
  if (end == lo) {
    sph[c] = make_float4(0.f, 0.f, 0.f, -3e38f);
    return;
  }
  const float cx = 0.5f * (mn[0] + mx[0]), cy = 0.5f * (mn[1] + mx[1]), cz = 0.5f * (mn[2] + mx[2]);
  float R = 0.f;
  for (uint64_t t = lo; t < end; ++t) {
    const float4 r = bp32[t];
    const float ex = r.x - cx, ey = r.y - cy, ez = r.z - cz;
    R = fmaxf(R, sqrtf(ex * ex + ey * ey + ez * ez) + r.w);
  }
  const float m = fmaxf(fabsf(cx), fmaxf(fabsf(cy), fabsf(cz))) + R;
  sph[c] = make_float4(cx, cy, cz, R * 1.000001f + 1e-6f * m);
}

// One thread per sorted position s: the inverse permutation and the
// particle's records in cell order -- the only gather of the state per list
// build; the candidate and narrow phases read bp / pk of neighbouring cells,
// which are neighbouring lines.
__global__ void k_cells(DevScene d, const uint32_t* __restrict__ ks, const uint32_t* __restrict__ is) {
  const uint64_t n = d.n;
  const uint64_t s = (uint64_t)blockIdx.x * blockDim.x + threadIdx.x;
  if (s >= n) return;
  const uint32_t i = is[s];
  d.rank[i] = (uint32_t)s;
  if (s == 0) {  // an order and its inverse stand; the next build counts its movers afresh
    d.sort_state[0] = 1u;
    d.sort_state[2] = 0u;
    d.nl[kNlStale] = 0u;
  }
  d.cand_count[s] = 0u;  // the half-shell search adds to it from both sides
  d.pend[s] = 0u;
  const uint32_t shp = d.shape[i];
  PoseRec r;
  r.x = d.pos[i];
  r.y = d.pos[n + i];
  r.z = d.pos[2 * n + i];
  r.qx = d.quat[i];
  r.qy = d.quat[n + i];
  r.qz = d.quat[2 * n + i];
  r.qw = d.quat[3 * n + i];
  r.shape = shp;
  r.sim = d.sim[i];
  d.pk[s] = r;
  VelRec v;
#pragma unroll
  for (int k = 0; k < 3; ++k) {
    v.v[k] = d.vel[k * n + i];
    v.w[k] = d.omega[k * n + i];
  }
  d.vk[s] = v;
  if (d.hk)
    for (int k = 0; k < 12; ++k) d.hk[12 * s + k] = d.ab_hist[k * n + i];
  if (d.nobs) d.rws[s] = d.np64[shp].rc_max;
  const double rc = d.rc_pf[shp];
  const SimGrid& g = d.sgrids[r.sim];
  const double reach = rc + g.half_skin;
  d.rcs[s] = rc;
  d.bp[s] = make_double4(r.x, r.y, r.z, reach);
  d.bp32[s] = make_float4((float)(r.x - g.lo[0]), (float)(r.y - g.lo[1]), (float)(r.z - g.lo[2]), (float)reach);
  const double p[3] = {r.x, r.y, r.z};
  uint32_t c[3];
  const SimGrid& gr = d.grids[r.sim];
  cell_of(gr, p, c);
  d.rkey[s] = cell_key(gr, c);
  // a centre outside a periodic side is folded into a border cell now and
  // wrapped by the step
  bool out = false;
#pragma unroll
  for (int k = 0; k < 3; ++k) out |= ((g.periodic >> k) & 1) && (p[k] < g.lo[k] || p[k] >= g.hi[k]);
  if (out) d.nl[kNlOutside] = 1u;
}

void launch_cells(const DevScene& d, const uint32_t* keys_s, const uint32_t* idx_s, hipStream_t s) {
  const uint64_t offs = (uint64_t)d.ncells + 1;
  if (d.n)  // the records first: the cell spheres are built from bp32
    hipLaunchKernelGGL(k_cells, dim3((unsigned)((d.n + kBlock - 1) / kBlock)), dim3(kBlock), 0, s, d, keys_s,
                       idx_s);
  // the cell spheres serve the per-particle candidate search only
  hipLaunchKernelGGL(k_cell_off, dim3((unsigned)((offs + kBlock - 1) / kBlock)), dim3(kBlock), 0, s, keys_s, d.bp32,
                     d.n, (uint64_t)d.ncells, d.cell_off, d.cand_staged || d.cand_half ? nullptr : d.cell_sph);
}

// ---- candidates -------------------------------------------------------------------
// The search finds the pairs whose list spheres overlap: prefilter radii
// grown by half the skin, so the lists hold every pair whose bounding spheres
// can overlap until some particle has moved by half the skin.  The steps
// apply the prefilter itself to them (narrow phase).  Without a skin the two
// are the same.
__device__ __forceinline__ void list_overflow(const DevScene& d, uint32_t over, uint32_t cnt) {
  if (over) d.nl[kNlOver] = 1u;
  if (!d.skin) {  // the lists are the step's candidates: an overflow is an error
    count_add(d.counters, kCntOverflow, over);
    count_max(d.counters, kCntMaxCand, over ? cnt : 0u);
  }
}

// One thread per sorted position s (spatially coherent waves).  Writes the
// sorted positions of its candidates, in the reference visit order, into
// cand[k * N + s] (k-major, so the lanes of a wave write neighbouring words)
// and their count into cand_count[s].  Residents of a cell ascend in sorted
// position exactly as in particle index (the sort is stable on an identity
// payload).  Each neighbour cell is its own loop: merging the three cells of
// a row into one range [off[c-1], off[c+2]) (they have consecutive keys) was
// measured 24 % slower on the 10^6 superquadric bed.
__device__ __forceinline__ void cand_scan(const DevScene& d, uint32_t t0, uint32_t t1, uint32_t s, V3<double> xi,
                                          double ri, const SimGrid& g, uint32_t& cnt, uint32_t& over) {
  const uint64_t n = d.n;
  for (uint32_t t = t0; t < t1; ++t) {
    if (t == s) continue;
    const double4 bj = d.bp[t];
    V3<double> dd = V3<double>{bj.x, bj.y, bj.z} - xi;
    if (g.periodic) dd = min_image(g, dd);
    const double rs = ri + bj.w;
    if (!(dd.x * dd.x + dd.y * dd.y + dd.z * dd.z < rs * rs * (1.0 + kPrefilterSlack))) continue;
    if (cnt < d.K)
      d.cand[(uint64_t)cnt * n + s] = t;
    else
      over = 1;
    ++cnt;
  }
}

// The 27 neighbour cells of cell `key` in the reference order (LinkedCell.cpp:
// 41-70: z outer, then y, then x): f(w, c) for each cell c inside the grid,
// periodic axes wrapped; w = (dz + 1) * 3 + (dy + 1) is the neighbour row.
template <class F>
__device__ __forceinline__ void for_each_neighbor(const SimGrid& g, uint32_t key, F&& f) {
  const int nx = (int)g.n3[0], ny = (int)g.n3[1], nz = (int)g.n3[2];
  const uint32_t local = key - g.base;
  const int cx = (int)(local % (uint32_t)nx);
  const int cy = (int)((local / (uint32_t)nx) % (uint32_t)ny);
  const int cz = (int)(local / ((uint32_t)nx * (uint32_t)ny));
  const bool px = g.periodic & 1, py = g.periodic & 2, pz = g.periodic & 4;
  for (int dz = -1; dz <= 1; ++dz) {
    int z = cz + dz;
    if (pz) z = z < 0 ? z + nz : (z >= nz ? z - nz : z);
    if (z < 0 || z >= nz) continue;
    for (int dy = -1; dy <= 1; ++dy) {
      int y = cy + dy;
      if (py) y = y < 0 ? y + ny : (y >= ny ? y - ny : y);
      if (y < 0 || y >= ny) continue;
      const int w = (dz + 1) * 3 + (dy + 1);
      const uint32_t row = g.base + ((uint32_t)z * (uint32_t)ny + (uint32_t)y) * (uint32_t)nx;
      for (int dx = -1; dx <= 1; ++dx) {
        int x = cx + dx;
        if (px) x = x < 0 ? x + nx : (x >= nx ? x - nx : x);
        if (x < 0 || x >= nx) continue;
        f(w, row + (uint32_t)x);
      }
    }
  }
}

// Every lane reads its neighbours' records from global memory (lanes of a
// cell read the same lines, which the caches serve).  A neighbour cell whose
// bounding sphere (cell_sph) is out of reach is skipped whole; the resident
// checks -- ~90 per particle on the superquadric bed, nearly all rejected --
// read the 16-byte FP32 records bp32 (positions relative to the sim's domain
// minimum) with a conservative test; every pair it passes is decided by the
// FP64 test of cand_scan, so the candidate lists are those of the FP64
// prefilter bit for bit.  The relative coordinates carry at most 2^-24 of
// their magnitude, the difference and the periodic shift as much again of
// theirs; the margin is 1e-6 of those magnitudes, several times the bound.
__global__ void __launch_bounds__(kBlock) k_candidates_direct(DevScene d, const uint32_t* __restrict__ ks) {
  const uint64_t n = d.n;
  const uint64_t s = (uint64_t)blockIdx.x * blockDim.x + threadIdx.x;
  uint32_t cnt = 0, over = 0;
  if (s < n) {
    const double4 bi = d.bp[s];
    const float4 fi = d.bp32[s];
    // one sim: no need to read the pose record (a 64-byte line) for its id
    const SimGrid g = d.sgrids[d.nsims > 1 ? d.pk[s].sim : 0u];
    const V3<double> xi = {bi.x, bi.y, bi.z};
    const bool px = g.periodic & 1, py = g.periodic & 2, pz = g.periodic & 4;
    const float Lx = (float)g.L[0], Ly = (float)g.L[1], Lz = (float)g.L[2];
    // periodic image by a reciprocal: it can pick another image than the
    // FP64 test only at separations near L/2, far beyond any candidate
    const float iLx = 1.f / Lx, iLy = 1.f / Ly, iLz = 1.f / Lz;
    const float base = fmaxf(fabsf(fi.x), fmaxf(fabsf(fi.y), fabsf(fi.z))) +
                       3.f * (g.periodic ? fmaxf(Lx, fmaxf(Ly, Lz)) : 0.f);
    // conservative FP32 reach test of a sphere q (centre, radius) from fi
    auto reach = [&](const float4& q) {
      float ex = q.x - fi.x, ey = q.y - fi.y, ez = q.z - fi.z;
      if (px) ex -= Lx * rintf(ex * iLx);
      if (py) ey -= Ly * rintf(ey * iLy);
      if (pz) ez -= Lz * rintf(ez * iLz);
      const float mq = fmaxf(fabsf(q.x), fmaxf(fabsf(q.y), fabsf(q.z)));
      const float rs = (fi.w + q.w) * 1.000001f + 1e-6f * (base + mq);
      return ex * ex + ey * ey + ez * ez < rs * rs;
    };
    // (loading a row's three spheres and offsets together was measured no
    // faster, at 78 instead of 64 VGPRs)
    for_each_neighbor(g, ks[s], [&](int, uint32_t c) {
      const float4 q = d.cell_sph[c];
      if (!(q.w >= 0.f && reach(q))) return;  // empty, or out of reach
      const uint32_t t1 = d.cell_off[c + 1];
      for (uint32_t t = d.cell_off[c]; t < t1; ++t) {
        if (t == (uint32_t)s) continue;
        if (reach(d.bp32[t])) cand_scan(d, t, t + 1, (uint32_t)s, xi, bi.w, g, cnt, over);
      }
    });
    d.cand_count[s] = cnt < d.K ? cnt : d.K;
  }
  list_overflow(d, over, cnt);
}

// Half shell.  The prefilter is symmetric -- the FP64 test of cand_scan
// takes x_j - x_i, its minimum image and r_i + r_j, and negating the
// difference or swapping the sum's operands changes no rounding -- so each
// unordered pair needs one test: a particle tests the residents after it in
// its own cell and those of the 13 cells that come after its own in one
// direction ((0, 0, +1), (0, +1, *), (+1, *, *) in (dz, dy, dx)), and every
// pair found goes into both particles' lists (k-major slots taken with an
// atomic on the list's count; cand_count is zeroed by k_cells).  Every pair
// of neighbouring cells is one cell's forward neighbour exactly once when
// each periodic axis has at least three cells (the host takes the full
// search otherwise).  The slots come in no fixed order; k_expand puts each
// list in the reference visit order.  Same resident test and FP64 decision
// as k_candidates_direct, so the lists are the same, with half the checks.
__device__ __forceinline__ void half_pair(const DevScene& d, uint32_t s, uint32_t t, V3<double> xi, double ri,
                                          const SimGrid& g, uint32_t& over) {
  const double4 bj = d.bp[t];
  V3<double> dd = V3<double>{bj.x, bj.y, bj.z} - xi;
  if (g.periodic) dd = min_image(g, dd);
  const double rs = ri + bj.w;
  if (!(dd.x * dd.x + dd.y * dd.y + dd.z * dd.z < rs * rs * (1.0 + kPrefilterSlack))) return;
  const uint64_t n = d.n;
  const uint32_t a = atomicAdd(&d.cand_count[s], 1u);
  if (a < d.K)
    d.cand[(uint64_t)a * n + s] = t;
  else
    over = 1;
  const uint32_t b = atomicAdd(&d.cand_count[t], 1u);
  if (b < d.K)
    d.cand[(uint64_t)b * n + t] = s;
  else
    over = 1;
}

// Half-shell search by cell: sixteen lanes per cell, four cells per wave.
// Lanes 0..13 of a cell's group take the cell itself and its 13 forward
// neighbour cells ((0, 0, +1), (0, +1, *), (+1, *, *) in (dz, dy, dx)), and a
// prefix sum of their resident counts lays the fourteen ranges of sorted
// positions end to end.  The cell's residents sit in LDS with the resident
// half of the reach bound; the group reads the list 16 records at a time,
// one per lane (the next 16 in flight meanwhile), shifted to the cell's
// periodic image of its range (so differences need no minimum image), and
// tests its record against the residents in LDS.  Pairs inside the cell are
// tested once (the lane's record after the resident).  Pairs the
// conservative FP32 test passes collect in the wave's LDS list; at the end
// (or when it fills) the wave takes them 64 at a time, one per lane, through
// the FP64 decision and the appends to both lists (half_pair), so it waits
// for the appends' atomics once, not once per hit.  A neighbourhood's records
// are read once per cell instead of once per resident, and the tests of a
// cell run side by side on the lanes instead of as one dependent chain per
// particle.  Dense cells (polydisperse beds, whose cell side follows the
// largest grain, hold tens to hundreds of the small ones) are shared by
// several groups: a cell of q residents gets C(q) x P(q) of them, group
// (c, p) taking the resident chunks c, c + C, ... and the p-th of P equal
// slices of the list, so the ~14 q records of a dense cell's list are
// tested by many waves side by side.  Each (resident, record) pair still
// falls to exactly one group.  The groups then come from a work list (a
// count per cell, its scan and the cells' group entries) walked by a grid
// of fixed size.
constexpr int kCellLanes = 16;
constexpr uint32_t kResLds = 32;   // residents of a cell held in LDS at a time
constexpr uint32_t kPairLds = 256; // pairs a wave collects before deciding them

// the FP32 reach test in two halves: a resident's a = w (1 + 1e-6) + 1e-6
// (max|x| + span) and a record's b = w (1 + 1e-6) + 1e-6 max|x|; pair (i, j)
// passes when |x_j - x_i| < a_i + b_j (the bound of k_candidates_direct, as
// a sum of two roundings: still ~1e-6 relative above the FP64 test's)
__device__ __forceinline__ float reach_half(const float4& q, float span) {
  return q.w * 1.000001f + 1e-6f * (fmaxf(fabsf(q.x), fmaxf(fabsf(q.y), fabsf(q.z))) + span);
}

// resident chunks and list slices of a cell of q residents (work-list
// mode): chunks of kResLds, and slices of about kListLds records (8 rounds
// of kCellLanes) of the ~14 q records of its list; C(q) P(q) <= q, so a bed
// has at most n groups
constexpr uint32_t kListLds = 128;  // list positions whose range index a group keeps in LDS
__device__ __forceinline__ uint32_t half_chunks(uint32_t q) { return min(8u, (q + kResLds - 1) / kResLds); }
__device__ __forceinline__ uint32_t half_slices(uint32_t q) {
  return max(1u, min(16u, (14u * min(q, 1u << 20) + kListLds - 1) / kListLds));
}

struct HalfLds {
  uint4 e[kBlock / kCellLanes][4], d[kBlock / kCellLanes][4];  // range starts in list order, list index -> sorted position
  uint32_t w[kBlock / kCellLanes][16];                        // range image shifts: 2 bits per axis (0, +L, -L)
  float4 res[kBlock / kCellLanes][kResLds];                   // residents (x, y, z, a)
  uint2 pair[kBlock / 64][kPairLds];                          // the wave's pairs to decide
  uint8_t rk[kBlock / kCellLanes][kListLds];                  // range of list position lo + i
};

// decide the wave's collected pairs, one per lane
template <bool MULTI>
__device__ __forceinline__ void half_decide(const DevScene& d, HalfLds& L, uint32_t& nw, uint32_t& over) {
  const uint32_t lane = __lane_id(), wv = threadIdx.x / 64;
  __builtin_amdgcn_fence(__ATOMIC_SEQ_CST, "workgroup");  // the wave's LDS writes are done
  for (uint32_t k = lane; k < nw; k += 64) {
    const uint2 p = L.pair[wv][k];
    const double4 bi = d.bp[p.x];
    const SimGrid& gp = d.sgrids[MULTI ? d.pk[p.x].sim : 0u];
    half_pair(d, p.x, p.y, V3<double>{bi.x, bi.y, bi.z}, bi.w, gp, over);
  }
  __builtin_amdgcn_fence(__ATOMIC_SEQ_CST, "workgroup");  // read before the list is refilled
  nw = 0;
}

// one group's share of cell c: its resident chunks chunk0, chunk0 + sc, ...
// against slice `slice` of sp of the list.  Every thread of the block calls
// it (a cell index >= ncells: an idle group).  The wave's pair list and its
// length nw carry over between calls.
template <bool MULTI>
__device__ __forceinline__ void half_group(const DevScene& d, HalfLds& L, uint64_t c, uint32_t chunk0,
                                           uint32_t slice, uint32_t sc, uint32_t sp, uint32_t& nw, uint32_t& over) {
  const uint32_t lane = __lane_id();
  const uint32_t sub = lane % kCellLanes;  // lane within the cell's group
  const int gb = (int)(lane - sub);        // the group's first lane
  const uint32_t grp = threadIdx.x / kCellLanes;
  const uint32_t wv = threadIdx.x / 64;
  uint32_t a0 = 0, a1 = 0;
  if (c < d.ncells) {
    a0 = d.cell_off[c];
    a1 = d.cell_off[c + 1];
  }
  const bool busy = a1 > a0;
  const SimGrid& g = d.sgrids[MULTI && busy ? d.pk[a0].sim : 0u];
  // lane k < 14 of the group: the k-th range (k = 0: the cell; 1: (0, 0, +1);
  // 2..4: (0, +1, -1..+1); 5..13: (+1, -1..+1, -1..+1)), [t0, t1), and the
  // image shift of a range reached across a periodic side
  uint32_t t0 = a0, t1 = sub == 0 ? a1 : a0, wc = 0;
  if (busy && sub > 0 && sub < 14) {
    const int nx = (int)g.n3[0], ny = (int)g.n3[1], nz = (int)g.n3[2];
    const uint32_t local = (uint32_t)c - g.base;
    const int cx = (int)(local % (uint32_t)nx);
    const int cy = (int)((local / (uint32_t)nx) % (uint32_t)ny);
    const int cz = (int)(local / ((uint32_t)nx * (uint32_t)ny));
    const int k = (int)sub;
    const int dz = k < 5 ? 0 : 1;
    const int dy = k == 1 ? 0 : (k < 5 ? 1 : (k - 5) / 3 - 1);
    const int dx = k == 1 ? 1 : (k < 5 ? k - 3 : (k - 5) % 3 - 1);
    int x = cx + dx, y = cy + dy, z = cz + dz;
    // a cell reached across the low side lies L beyond it: its records shift by -L
    auto wrap = [&](int& v, int nv, bool per, int bit) {
      if (!per) return;
      if (v < 0) {
        v += nv;
        wc |= 2u << bit;
      } else if (v >= nv) {
        v -= nv;
        wc |= 1u << bit;
      }
    };
    wrap(x, nx, g.periodic & 1, 0);
    wrap(y, ny, g.periodic & 2, 2);
    wrap(z, nz, g.periodic & 4, 4);
    if (x >= 0 && x < nx && y >= 0 && y < ny && z >= 0 && z < nz) {
      const uint32_t cn = g.base + ((uint32_t)z * (uint32_t)ny + (uint32_t)y) * (uint32_t)nx + (uint32_t)x;
      t0 = d.cell_off[cn];
      t1 = d.cell_off[cn + 1];
    }
  }
  const uint32_t cnt = t1 - t0;
  uint32_t incl = cnt;
#pragma unroll
  for (int o = 1; o < kCellLanes; o <<= 1) {
    const uint32_t y = __shfl_up(incl, o, kCellLanes);
    if (sub >= (uint32_t)o) incl += y;
  }
  ((uint32_t*)L.e[grp])[sub] = sub < 14 ? incl - cnt : 0xffffffffu;
  ((uint32_t*)L.d[grp])[sub] = t0 - (incl - cnt);
  L.w[grp][sub] = wc;
  const uint32_t m = __shfl(incl, gb + 13);  // the list's length
  // this group's slice [lo, hi) of the list, whole rounds of kCellLanes
  const uint32_t slen = (((m + sp - 1) / sp) + kCellLanes - 1) / kCellLanes * kCellLanes;
  const uint32_t lo = min(m, slice * slen), hi = min(m, lo + slen);
  // each range's lane writes its index at its positions of the slice (the
  // first kListLds of them), so a round finds a position's range with one
  // LDS byte instead of comparing against the 14 range starts
  {
    const uint32_t p0 = max(incl - cnt, lo), p1 = min(incl, min(hi, lo + kListLds));
    for (uint32_t p = p0; p < p1; ++p) L.rk[grp][p - lo] = (uint8_t)sub;
  }
  const float Lx = (float)g.L[0], Ly = (float)g.L[1], Lz = (float)g.L[2];
  const float span = 3.f * (g.periodic ? fmaxf(Lx, fmaxf(Ly, Lz)) : 0.f);
  // list index -> (sorted position, range): from the range bytes within
  // the first kListLds positions of the slice, past them by comparing with
  // the range starts (a slice longer than kListLds: a dense cell outside
  // the work list)
  auto locate = [&](uint32_t idx, uint32_t& t, uint32_t& k) {
    if (idx < hi && idx - lo < kListLds) {
      k = L.rk[grp][idx - lo];
      t = idx + ((const uint32_t*)L.d[grp])[k];
      return;
    }
#pragma unroll
    for (int w = 0; w < 4; ++w) {
      const uint4 e4 = L.e[grp][w], d4 = L.d[grp][w];
      if (w == 0 || idx >= e4.x) t = idx + d4.x, k = 4 * w;
      if (idx >= e4.y) t = idx + d4.y, k = 4 * w + 1;
      if (idx >= e4.z) t = idx + d4.z, k = 4 * w + 2;
      if (idx >= e4.w) t = idx + d4.w, k = 4 * w + 3;
    }
  };
  const uint32_t na = a1 - a0;
  // the residents r0 .. r0 + nr - 1 of the cell into LDS (read by this group only)
  auto stage = [&](uint32_t r0, uint32_t nr) {
    for (uint32_t r = sub; r < nr; r += kCellLanes) {
      float4 q = d.bp32[a0 + r0 + r];
      q.w = reach_half(q, span);
      L.res[grp][r] = q;
    }
  };
  const uint32_t rfirst = chunk0 * kResLds, rstep = sc * kResLds;
  // (lanes without a record read position q0: a0 can be n past the last cell)
  const uint32_t q0 = busy ? a0 : 0u;
  uint32_t tn = 0, kn = 0;
  float4 qn;
  stage(rfirst, na > rfirst ? min(na - rfirst, kResLds) : 0u);
  __syncthreads();  // the range tables and the first chunk
  for (uint32_t r0 = rfirst; __any(r0 < na); r0 += rstep) {
    const uint32_t nr = na > r0 ? min(na - r0, kResLds) : 0u;  // residents in this chunk
    if (r0 > rfirst) {  // a cell of more than kResLds residents: the next chunk
      stage(r0, nr);
      __builtin_amdgcn_fence(__ATOMIC_SEQ_CST, "workgroup");
    }
    locate(lo + sub, tn, kn);
    qn = d.bp32[lo + sub < hi && nr > 0 ? tn : q0];
    const uint32_t first = a0 + r0;
    const uint32_t jw = (uint32_t)__builtin_amdgcn_readfirstlane((int)wave_max(nr));  // the loop's bound
    for (uint32_t b0 = lo; __any(b0 < hi); b0 += kCellLanes) {
      const uint32_t idx = b0 + sub;
      const bool live = idx < hi && nr > 0;
      const uint32_t t = tn, k = kn;
      float4 q = qn;
      // the next round's record, in flight during this round's tests (the
      // range tables are read from LDS each round: the compiler barrier
      // keeps them from being hoisted into 32 loop-long VGPRs)
      asm volatile("" ::: "memory");
      locate(idx + kCellLanes, tn, kn);
      qn = d.bp32[idx + kCellLanes < hi && nr > 0 ? tn : q0];
      const float b = reach_half(q, 0.f);
      const uint32_t w = L.w[grp][k];
      q.x += (w & 1u) ? Lx : ((w & 2u) ? -Lx : 0.f);
      q.y += (w & 4u) ? Ly : ((w & 8u) ? -Ly : 0.f);
      q.z += (w & 16u) ? Lz : ((w & 32u) ? -Lz : 0.f);
      // residents j < jmax of the chunk pair with the lane's record: all of
      // them, or in the cell itself those before the record
      const uint32_t jmax = !live ? 0u : (k > 0 ? nr : (t > first ? min(t - first, nr) : 0u));
      uint32_t mask = 0;
#pragma unroll 4
      for (uint32_t j = 0; j < jw; ++j) {
        const float4 f = L.res[grp][j];
        const float ex = q.x - f.x, ey = q.y - f.y, ez = q.z - f.z;
        const float rs = f.w + b;
        mask |= (uint32_t)(ex * ex + ey * ey + ez * ez < rs * rs) << j;
      }
      mask &= jmax >= 32u ? ~0u : (1u << jmax) - 1u;  // residents j < jmax only
      // the lanes' pairs into the wave's list, one per lane at a time
      while (__any(mask != 0)) {
        const bool has = mask != 0;
        const uint64_t bal = __ballot(has);
        const uint32_t nb = (uint32_t)__popcll(bal);
        if (nw + nb > kPairLds) half_decide<MULTI>(d, L, nw, over);
        if (has) {
          const uint32_t pos =
              nw + __builtin_amdgcn_mbcnt_hi((uint32_t)(bal >> 32), __builtin_amdgcn_mbcnt_lo((uint32_t)bal, 0u));
          L.pair[wv][pos] = make_uint2(first + (uint32_t)(__ffs(mask) - 1), t);
          mask &= mask - 1;
        }
        nw += nb;
      }
    }
  }
}

// one group per cell (beds of a few particles per cell)
template <bool MULTI>
__global__ void __launch_bounds__(kBlock) k_candidates_half(DevScene d) {
  __shared__ HalfLds L;
  uint32_t nw = 0, over = 0;  // nw: pairs in the wave's LDS list (wave-uniform)
  const uint64_t c = ((uint64_t)blockIdx.x * blockDim.x + threadIdx.x) / kCellLanes;
  half_group<MULTI>(d, L, c, 0u, 0u, 1u, 1u, nw, over);
  if (nw) half_decide<MULTI>(d, L, nw, over);
  list_overflow(d, over, 0u);
}

// the work list: groups per cell, their exclusive scan (half_goff, total at
// [ncells]) and each group's cell (half_glist)
__global__ void k_half_work(DevScene d) {
  const uint64_t c = (uint64_t)blockIdx.x * blockDim.x + threadIdx.x;
  if (c >= d.ncells) return;
  const uint32_t q = d.cell_off[c + 1] - d.cell_off[c];
  d.half_goff[c] = q ? half_chunks(q) * half_slices(q) : 0u;
}

__global__ void k_half_list(DevScene d) {
  const uint64_t c = (uint64_t)blockIdx.x * blockDim.x + threadIdx.x;
  if (c >= d.ncells) return;
  const uint32_t o = d.half_goff[c], e = d.half_goff[c + 1];
  for (uint32_t k = o; k < e && k < (uint32_t)d.n; ++k) d.half_glist[k] = (uint32_t)c;
}

// groups from the work list, gridDim.x x 16 of them at a time
template <bool MULTI>
__global__ void __launch_bounds__(kBlock) k_candidates_half_wl(DevScene d) {
  __shared__ HalfLds L;
  constexpr uint32_t G = kBlock / kCellLanes;
  const uint32_t total = min(d.half_goff[d.ncells], (uint32_t)d.n);
  const uint32_t grp = threadIdx.x / kCellLanes;
  uint32_t nw = 0, over = 0;
  for (uint32_t base = blockIdx.x * G; base < total; base += gridDim.x * G) {  // block-uniform
    const uint32_t gi = base + grp;
    uint64_t c = d.ncells;
    uint32_t part = 0, sc = 1, sp = 1;
    if (gi < total) {
      c = d.half_glist[gi];
      part = gi - d.half_goff[c];
      const uint32_t q = d.cell_off[c + 1] - d.cell_off[c];
      sc = half_chunks(q);
      sp = half_slices(q);
    }
    half_group<MULTI>(d, L, c, part / sp, part % sp, sc, sp, nw, over);
  }
  if (nw) half_decide<MULTI>(d, L, nw, over);
  list_overflow(d, over, 0u);
}

// The block's neighbour records are staged in LDS first.  The block holds
// consecutive sorted positions, so its keys span [kmin, kmax] and the cells
// its lanes visit in neighbour row (dz, dy) lie in the key window
// [kmin + o - 1, kmax + o + 1], o = (dz ny + dy) nx: nine windows, each a
// contiguous range of sorted positions [off[lo], off[hi + 1]), read once,
// coalesced, instead of once per visiting lane.  Records are kept in FP32
// relative to the block's first particle (16 B); a lane's cell whose range
// lies inside its row's window is scanned from LDS with a conservative FP32
// test, and every pair the FP32 test passes is decided by the FP64 test of
// cand_scan, so the candidate lists are those of the FP64 prefilter bit for
// bit.  Cells outside the windows (periodic wraps, a block spanning sims,
// windows beyond the LDS capacity) are scanned from global memory.  It pays
// off when cells hold many particles (long scans per lane); with a few per
// cell the direct kernel, at twice the occupancy, is faster.
constexpr int kCandStage = 2520;  // staged records per block: 4 blocks per CU in 160 KB of LDS

__global__ void __launch_bounds__(kBlock) k_candidates_staged(DevScene d, const uint32_t* __restrict__ ks) {
  __shared__ float4 stage[kCandStage];
  __shared__ uint32_t w_lo[9], w_hi[9], w_base[10];
  __shared__ uint32_t vmax_bits;
  __shared__ double org[3];
  const uint64_t n = d.n;
  const uint64_t b0 = (uint64_t)blockIdx.x * blockDim.x;
  const uint64_t s = b0 + threadIdx.x;
  if (threadIdx.x < 9) {
    const uint64_t last = b0 + blockDim.x - 1 < n ? b0 + blockDim.x - 1 : n - 1;
    const SimGrid& g0 = d.sgrids[d.pk[b0].sim];
    const int64_t dz = (int64_t)(threadIdx.x / 3) - 1, dy = (int64_t)(threadIdx.x % 3) - 1;
    const int64_t o = (dz * (int64_t)g0.n3[1] + dy) * (int64_t)g0.n3[0];
    int64_t lo = (int64_t)ks[b0] + o - 1, hi = (int64_t)ks[last] + o + 1;
    lo = lo < 0 ? 0 : lo;
    hi = hi > (int64_t)d.ncells - 1 ? (int64_t)d.ncells - 1 : hi;
    uint32_t plo = 0, phi = 0;
    if (lo <= hi) {
      plo = d.cell_off[lo];
      phi = d.cell_off[hi + 1];
    }
    w_lo[threadIdx.x] = plo;
    w_hi[threadIdx.x] = phi;
  }
  if (threadIdx.x == 0) {
    vmax_bits = 0u;
    const double4 q = d.bp[b0];
    org[0] = q.x;
    org[1] = q.y;
    org[2] = q.z;
  }
  __syncthreads();
  if (threadIdx.x == 0) {  // greedy: windows in order while they fit
    uint32_t tot = 0;
    for (int w = 0; w < 9; ++w) {
      const uint32_t sz = w_hi[w] - w_lo[w];
      w_base[w] = tot;
      if (tot + sz <= (uint32_t)kCandStage)
        tot += sz;
      else
        w_hi[w] = w_lo[w];  // not staged: its cells are read from global memory
    }
    w_base[9] = tot;
  }
  __syncthreads();
  {
    const uint32_t tot = w_base[9];
    float vm = 0.f;
    int w = 0;
    for (uint32_t k = threadIdx.x; k < tot; k += blockDim.x) {
      while (k >= w_base[w + 1]) ++w;
      const double4 q = d.bp[w_lo[w] + (k - w_base[w])];
      const float4 r = make_float4((float)(q.x - org[0]), (float)(q.y - org[1]), (float)(q.z - org[2]), (float)q.w);
      stage[k] = r;
      vm = fmaxf(vm, fmaxf(fabsf(r.x), fmaxf(fabsf(r.y), fabsf(r.z))));
    }
    atomicMax(&vmax_bits, __float_as_uint(vm));  // non-negative floats order as their bits
  }
  __syncthreads();
  uint32_t cnt = 0, over = 0;
  if (s < n) {
    const double4 bi = d.bp[s];
    const SimGrid g = d.sgrids[d.pk[s].sim];
    const V3<double> xi = {bi.x, bi.y, bi.z};
    const double ri = bi.w;
    const bool px = g.periodic & 1, py = g.periodic & 2, pz = g.periodic & 4;
    // the FP32 test: relative coordinates carry at most 2^-24 of their
    // magnitude (bounded by the staged maximum and the lane's own), the
    // difference and the periodic shift as much again of theirs; the margin
    // is 1e-6 of those magnitudes, several times the bound
    const float xf = (float)(xi.x - org[0]), yf = (float)(xi.y - org[1]), zf = (float)(xi.z - org[2]);
    const float Lx = (float)g.L[0], Ly = (float)g.L[1], Lz = (float)g.L[2];
    const float Lw = g.periodic ? fmaxf(Lx, fmaxf(Ly, Lz)) : 0.f;
    const float mi = fmaxf(fabsf(xf), fmaxf(fabsf(yf), fabsf(zf)));
    const float margin = 1e-6f * (__uint_as_float(vmax_bits) + mi + 3.f * Lw);
    const float rif = (float)ri;
    for_each_neighbor(g, ks[s], [&](int w, uint32_t c) {
      const uint32_t wlo = w_lo[w], whi = w_hi[w];
      const uint32_t t0 = d.cell_off[c], t1 = d.cell_off[c + 1];
      if (t0 >= wlo && t1 <= whi) {
        const uint32_t sb = w_base[w] - wlo;  // index t + sb (mod 2^32) = w_base[w] + (t - wlo)
        for (uint32_t t = t0; t < t1; ++t) {
          if (t == (uint32_t)s) continue;
          const float4 r = stage[t + sb];
          float ex = r.x - xf, ey = r.y - yf, ez = r.z - zf;
          if (px) ex -= Lx * rintf(ex / Lx);
          if (py) ey -= Ly * rintf(ey / Ly);
          if (pz) ez -= Lz * rintf(ez / Lz);
          const float rs = (rif + r.w) * 1.000001f + margin;
          if (!(ex * ex + ey * ey + ez * ez < rs * rs)) continue;
          cand_scan(d, t, t + 1, (uint32_t)s, xi, ri, g, cnt, over);
        }
      } else {
        cand_scan(d, t0, t1, (uint32_t)s, xi, ri, g, cnt, over);
      }
    });
    d.cand_count[s] = cnt < d.K ? cnt : d.K;
  }
  list_overflow(d, over, cnt);
}

void launch_candidates(const DevScene& d, const uint32_t* keys_s, hipStream_t s) {
  const dim3 grid((unsigned)((d.n + d.block - 1) / d.block)), block(d.block);
  if (d.cand_staged)
    hipLaunchKernelGGL(k_candidates_staged, grid, block, 0, s, d, keys_s);
  else if (d.cand_half && d.half_wl) {
    const dim3 cb((unsigned)((d.ncells + kBlock - 1) / kBlock));
    hipLaunchKernelGGL(k_half_work, cb, dim3(kBlock), 0, s, d);
    launch_scan(d.half_goff, d.half_goff, d.ncells, d.scan_blocks, s);
    hipLaunchKernelGGL(k_half_list, cb, dim3(kBlock), 0, s, d);
    // at most n groups; 2,048 blocks of 16 keep every CU busy
    const uint64_t nb = (d.n + kBlock / kCellLanes - 1) / (kBlock / kCellLanes);
    const dim3 wg((unsigned)(nb < 2048 ? nb : 2048));
    if (d.nsims > 1)
      hipLaunchKernelGGL(k_candidates_half_wl<true>, wg, dim3(kBlock), 0, s, d);
    else
      hipLaunchKernelGGL(k_candidates_half_wl<false>, wg, dim3(kBlock), 0, s, d);
  } else if (d.cand_half) {
    const dim3 cg((unsigned)(((uint64_t)d.ncells * kCellLanes + kBlock - 1) / kBlock));
    if (d.nsims > 1)
      hipLaunchKernelGGL(k_candidates_half<true>, cg, dim3(kBlock), 0, s, d);
    else
      hipLaunchKernelGGL(k_candidates_half<false>, cg, dim3(kBlock), 0, s, d);
  }
  else
    hipLaunchKernelGGL(k_candidates_direct, grid, block, 0, s, d, keys_s);
}

// flat entry list in sorted positions: entry e = entry_off[s] + k.  Each list
// is put in the reference visit order of the positions it was built from --
// the 27 neighbour cells z outer, y, x inner, ascending id within a cell
// (LinkedCell.cpp:41-70, ComponentManagerCPU.cpp:364-421; cells further away,
// which a skin can reach, where their clamped offset puts them) -- by a
// sorting network over (slot, id).  Counts beyond K (an overflow) are clamped
// as the scan clamps them.
// Batcher's odd-even merge sort of kSortNet keys, ascending; every index a
// compile-time constant once the loops unroll, so the keys stay in registers.
// Lists of up to 16 keys take the 16-key network, up to 32 the 32-key one
// (32-bit keys, up to 2^27 particles: the slot above the id), longer ones
// rank each candidate.
constexpr int kSortNet = 16;
template <int N, class K>
__device__ __forceinline__ void sort_network(K (&key)[N]) {
#pragma unroll
  for (int p = 1; p < N; p <<= 1)
#pragma unroll
    for (int k = p; k >= 1; k >>= 1)
#pragma unroll
      for (int j = k % p; j + k < N; j += 2 * k)
#pragma unroll
        for (int i = 0; i < k; ++i)
          if (i + j + k < N && (i + j) / (2 * p) == (i + j + k) / (2 * p)) {
            const K a = key[i + j], b = key[i + j + k];
            key[i + j] = a < b ? a : b;
            key[i + j + k] = a < b ? b : a;
          }
}

__global__ void k_expand(DevScene d) {
  const uint64_t n = d.n;
  const uint32_t* cand = d.cand;
  const uint64_t s = (uint64_t)blockIdx.x * blockDim.x + threadIdx.x;
  if (s == 0) {
    // with a skin: no use when a list is cut, or when a centre lies outside a
    // periodic side, whose neighbours are those of the reference's border cell
    const uint32_t no_use = !d.skin ? 0u : (d.nl[kNlOver] ? 2u : (d.nl[kNlOutside] ? 3u : 0u));
    d.nl[kNlValid] = no_use ? 0u : (d.skin ? 1u : 2u);
    if (no_use) d.nl[kNlOver] = no_use;
  }
  uint32_t raw = 0;
  if (s < n) {
    raw = d.cand_count[s];
    const uint32_t c = raw < d.K ? raw : d.K;
    const uint32_t e0 = d.entry_off[s];
    const uint32_t id = d.sidx[s];
    if (d.warm) d.ws_nb[(uint64_t)(*d.ws_par) * n + id] = make_uint2(e0, c);
    const SimGrid& g = d.grids[d.nsims > 1 ? d.pk[s].sim : 0u];
    const uint32_t nx = g.n3[0], ny = g.n3[1];
    auto cell = [&](uint32_t key, int* o) {
      const uint32_t l = key - g.base;
      o[0] = (int)(l % nx);
      o[1] = (int)((l / nx) % ny);
      o[2] = (int)(l / (nx * ny));
    };
    int ci[3];
    cell(d.rkey[s], ci);
    auto order = [&](uint32_t t) -> uint64_t {
      int cj[3], v[3];
      cell(d.rkey[t], cj);
#pragma unroll
      for (int k = 0; k < 3; ++k) {
        int x = cj[k] - ci[k];
        const int m = (int)g.n3[k];
        if ((g.periodic >> k) & 1) x = 2 * x > m ? x - m : (2 * x < -m ? x + m : x);
        v[k] = x > 1 ? 1 : (x < -1 ? -1 : x);
      }
      return ((uint64_t)(uint32_t)(((v[2] + 1) * 3 + v[1] + 1) * 3 + v[0] + 1) << 32) | d.sidx[t];
    };
    constexpr uint32_t kId27 = (1u << 27) - 1u;
    auto net = [&](auto& key) {
      using K = typename std::decay<decltype(key[0])>::type;
      constexpr int N = (int)(sizeof(key) / sizeof(key[0]));
#pragma unroll
      for (int k = 0; k < N; ++k) {
        K v = ~(K)0;
        if ((uint32_t)k < c) {
          const uint64_t o = order(cand[(uint64_t)k * n + s]);
          v = sizeof(K) == 4 ? (K)(((o >> 32) << 27) | (o & kId27)) : (K)o;
        }
        key[k] = v;
      }
      sort_network<N>(key);
#pragma unroll
      for (int k = 0; k < N; ++k)
        if ((uint32_t)k < c) {
          d.pair_i[e0 + k] = (uint32_t)s;
          d.pair_j[e0 + k] = d.rank[sizeof(K) == 4 ? (uint32_t)key[k] & kId27 : (uint32_t)key[k]];
        }
    };
    if (c <= kSortNet) {
      uint64_t key[kSortNet];
      net(key);
    } else if (c <= 2 * kSortNet && n <= (1ull << 27)) {
      uint32_t key[2 * kSortNet];
      net(key);
    } else {
      // a long list: each candidate at its rank
      for (uint32_t k = 0; k < c; ++k) {
        const uint32_t tk = cand[(uint64_t)k * n + s];
        const uint64_t ok = order(tk);
        uint32_t rank = 0;
        for (uint32_t j = 0; j < c; ++j) rank += j != k && order(cand[(uint64_t)j * n + s]) < ok;
        d.pair_i[e0 + rank] = (uint32_t)s;
        d.pair_j[e0 + rank] = tk;
      }
    }
  }
  if (!d.skin) count_max(d.counters, kCntMaxCand, raw > d.K ? raw : 0u);
}

// Warm starts: each new entry takes the record its pair had in the lists
// before (the same slot first: a particle's list keeps its order while its
// neighbours stay, then the others, four loads in flight), or none.
__global__ void __launch_bounds__(kBlock) k_warm_carry(DevScene d) {
  const uint64_t n = d.n, KN = (uint64_t)d.K * n;
  const uint32_t E = d.entry_off[n];
  const uint32_t cur = *d.ws_par;
  const float4* old = d.ws + (uint64_t)(1u - cur) * KN;
  float4* now = d.ws + (uint64_t)cur * KN;
  const uint64_t stride = (uint64_t)gridDim.x * blockDim.x;
  for (uint64_t e = (uint64_t)blockIdx.x * blockDim.x + threadIdx.x; e < E; e += stride) {
    const uint32_t s = d.pair_i[e];
    const uint32_t wj = d.sidx[d.pair_j[e]];
    const uint2 nb = d.ws_nb[(uint64_t)(1u - cur) * n + d.sidx[s]];
    const uint32_t wk = (uint32_t)e - d.entry_off[s];
    const float4* pr = old + nb.x;
    float4 r = make_float4(0.f, 0.f, 0.f, 0.f);
    bool hit = false;
    if (wk < nb.y) {
      r = pr[wk];
      hit = __float_as_uint(r.w) == wj;
    }
    for (uint32_t k0 = 0; !hit && k0 < nb.y; k0 += 4) {
      float4 q[4];
#pragma unroll
      for (uint32_t u = 0; u < 4; ++u) q[u] = k0 + u < nb.y ? pr[k0 + u] : make_float4(0.f, 0.f, 0.f, 0.f);
#pragma unroll
      for (uint32_t u = 0; u < 4; ++u)
        if (!hit && k0 + u < nb.y && __float_as_uint(q[u].w) == wj) {
          r = q[u];
          hit = true;
        }
    }
    if (!hit) r = make_float4(0.f, 0.f, 0.f, 0.f);
    r.w = __uint_as_float(wj);
    now[e] = r;
    d.pair_flag[e] = kFlagCand;  // a record that may have to be forgotten
  }
}

void launch_expand(const DevScene& d, hipStream_t s) {
  const dim3 grid((unsigned)((d.n + d.block - 1) / d.block)), block(d.block);
  hipLaunchKernelGGL(k_expand, grid, block, 0, s, d);
  if (d.warm) hipLaunchKernelGGL(k_warm_carry, dim3((unsigned)cu_count() * 8), dim3(kBlock), 0, s, d);
}

// ---- the step's pairs, read out -----------------------------------------------------
// The entries flagged `want`, particle by particle (by id), each one's by
// (neighbour cell in the visit order, id) at the positions of the step: the
// lists' own order, unless one of them is in another cell than when the lists
// were built.  Between two steps, in arrays that only a step or a build fills.
__global__ void __launch_bounds__(kBlock) k_pair_count(DevScene d, uint32_t want, uint32_t* __restrict__ count) {
  const uint64_t i = (uint64_t)blockIdx.x * blockDim.x + threadIdx.x;
  if (i >= d.n) return;
  const uint32_t s = d.rank[i];
  uint32_t c = 0;
  for (uint32_t e = d.entry_off[s]; e < d.entry_off[s + 1]; ++e) c += (d.pair_flag[e] & want) != 0;
  count[i] = c;
}
__global__ void __launch_bounds__(kBlock) k_pair_list(DevScene d, uint32_t want, const uint32_t* __restrict__ off,
                                                      uint32_t* __restrict__ nb) {
  const uint64_t i = (uint64_t)blockIdx.x * blockDim.x + threadIdx.x;
  if (i >= d.n) return;
  const uint32_t s = d.rank[i], e0 = d.entry_off[s], e1 = d.entry_off[s + 1];
  const SimGrid& g = d.grids[d.sim[i]];
  uint32_t k = off[i];
  bool again = d.rkey[s] != d.key[i];
  for (uint32_t e = e0; e < e1; ++e) {
    if (!(d.pair_flag[e] & want)) continue;
    const uint32_t t = d.pair_j[e], j = d.sidx[t];
    again |= d.rkey[t] != d.key[j];
    nb[k++] = j;
  }
  if (!again) return;
  auto cell = [&](uint32_t key, uint32_t* c) {
    const uint32_t l = key - g.base;
    c[0] = l % g.n3[0];
    c[1] = (l / g.n3[0]) % g.n3[1];
    c[2] = l / (g.n3[0] * g.n3[1]);
  };
  uint32_t ci[3];
  cell(d.key[i], ci);
  auto order = [&](uint32_t e) -> uint64_t {
    const uint32_t j = d.sidx[d.pair_j[e]];
    uint32_t cj[3];
    cell(d.key[j], cj);
    return ((uint64_t)(uint32_t)cell_slot(g, ci, cj) << 32) | j;
  };
  for (uint32_t e = e0; e < e1; ++e) {
    if (!(d.pair_flag[e] & want)) continue;
    const uint64_t me = order(e);
    uint32_t place = off[i];
    for (uint32_t f = e0; f < e1; ++f) place += (d.pair_flag[f] & want) && order(f) < me;
    nb[place] = (uint32_t)me;
  }
}
PairLists launch_pair_lists(const DevScene& d, uint32_t want, bool list, hipStream_t s) {
  const dim3 grid((unsigned)((d.n + kBlock - 1) / kBlock));
  hipLaunchKernelGGL(k_pair_count, grid, dim3(kBlock), 0, s, d, want, d.obs_list2);
  launch_scan(d.obs_list2, d.obs_list, d.n, d.scan_blocks, s);
  if (list) hipLaunchKernelGGL(k_pair_list, grid, dim3(kBlock), 0, s, d, want, d.obs_list, d.cand);
  return {d.obs_list, d.cand};
}

int cu_count() {
  static int cus = 0;
  if (!cus) {
    int dev = 0, c = 0;
    if (hipGetDevice(&dev) == hipSuccess &&
        hipDeviceGetAttribute(&c, hipDeviceAttributeMultiprocessorCount, dev) == hipSuccess && c > 0)
      cus = c;
    else
      cus = 256;
  }
  return cus;
}

}  // namespace gr
