// gr_narrow.hpp -- per-entry narrow phase + contact force, per-particle
// reduction + walls + gravity + explicit integration, and the standalone GJK
// batch.  Included by gr_narrow64.hip (T = double, built without FMA
// contraction) and gr_narrow32.hip (T = float, FP32-mixed).
#pragma once

#include <algorithm>
#include <type_traits>

#include "gr_internal.hpp"
#include "gr_move.hpp"

namespace gr {

template <class T> __device__ __forceinline__ const ShapeNP<T>* np_table(const DevScene& d);
template <> __device__ __forceinline__ const ShapeNP<double>* np_table<double>(const DevScene& d) { return d.np64; }
template <> __device__ __forceinline__ const ShapeNP<float>* np_table<float>(const DevScene& d) { return d.np32; }
template <class T> __device__ __forceinline__ const T* vt_full(const DevScene& d);
template <> __device__ __forceinline__ const double* vt_full<double>(const DevScene& d) { return d.verts64; }
template <> __device__ __forceinline__ const float* vt_full<float>(const DevScene& d) { return d.verts32; }
template <class T> __device__ __forceinline__ const T* vt_core(const DevScene& d);
template <> __device__ __forceinline__ const double* vt_core<double>(const DevScene& d) { return d.cverts64; }
template <> __device__ __forceinline__ const float* vt_core<float>(const DevScene& d) { return d.cverts32; }
template <class T> __device__ __forceinline__ const HookeP<T>* hk_table(const DevScene& d);
template <> __device__ __forceinline__ const HookeP<double>* hk_table<double>(const DevScene& d) { return d.hooke64; }
template <> __device__ __forceinline__ const HookeP<float>* hk_table<float>(const DevScene& d) { return d.hooke32; }

// Poses of A and B for the narrow phase.  FP64: world coordinates, with B's
// periodic image placed next to A exactly as the oracle does.  FP32: a frame
// translated to A's centre, B's offset taken in FP64 before rounding.
// dm: from A's centre to B's nearest image.  (The form below repeats the
// body: calling this one from it changes which products the compiler
// contracts in the FP32 search that follows, and so its results' last bits.)
template <class T>
__device__ __forceinline__ void pair_frames(V3<double> xi, Qt<double> qi, V3<double> xj, Qt<double> qj,
                                            V3<double> dm, Tr<T>& a2w, Tr<T>& b2w) {
  if constexpr (sizeof(T) == 8) {
    a2w.R = rot(qi);
    a2w.o = xi;
    b2w.R = rot(qj);
    b2w.o = same(dm, xj - xi) ? xj : xi + dm;
  } else {
    a2w.R = cvt<float>(rot(qi));
    a2w.o = {0.0f, 0.0f, 0.0f};
    b2w.R = cvt<float>(rot(qj));
    b2w.o = cvt<float>(dm);
  }
}
template <class T>
__device__ __forceinline__ void pair_frames(const SimGrid& g, V3<double> xi, Qt<double> qi, V3<double> xj,
                                            Qt<double> qj, Tr<T>& a2w, Tr<T>& b2w) {
  V3<double> dd = xj - xi;
  V3<double> dm = g.periodic ? min_image(g, dd) : dd;
  if constexpr (sizeof(T) == 8) {
    a2w.R = rot(qi);
    a2w.o = xi;
    b2w.R = rot(qj);
    b2w.o = same(dm, dd) ? xj : xi + dm;
  } else {
    a2w.R = cvt<float>(rot(qi));
    a2w.o = {0.0f, 0.0f, 0.0f};
    b2w.R = cvt<float>(rot(qj));
    b2w.o = cvt<float>(dm);
  }
}

// The GJK direction of the entry's last step (world frame), read only when
// the pair reaches GJK; a zero direction: none.
struct WarmLookup {
  const float4* rec;
  GR_D bool fetch(V3<float>& w) const {
    const float4 r = *rec;
    w = {r.x, r.y, r.z};
    const float nn = dot(w, w);
    return nn > 0.f && nn < INFINITY;
  }
};

// a rounded product: the FP32 unit is built with FMA contraction, which would
// fold it into the sum it goes into
__device__ __forceinline__ double product(double a, double b) {
  double p = a * b;
  asm("" : "+v"(p));
  return p;
}

// A sim's grid through the scalar cache (a wave-uniform address; grids do
// not change while kernels run).
__device__ __forceinline__ SimGrid uniform_grid(const SimGrid* p) {
  const auto* w = (const __attribute__((address_space(4))) uint32_t*)p;
  uint32_t v[sizeof(SimGrid) / 4];
#pragma unroll
  for (uint32_t k = 0; k < sizeof(SimGrid) / 4; ++k) v[k] = w[k];
  SimGrid g;
  __builtin_memcpy(&g, v, sizeof(g));
  return g;
}

// The bounding-sphere prefilter of the reference's particle loop
// (ComponentManagerCPU.cpp:384-396) for a list entry at the current
// positions: spheres overlapping, particles in neighbouring cells.  FP64
// without contraction in both precisions.  Spheres that overlap by less than
// a cell's side lie in neighbouring cells (any cell is at least that wide
// unless the caller asked for smaller ones), so the cells are worked out only
// for offsets within rounding of the side or more, and when a centre lay
// outside a periodic side (`outside`: its cell is a folded one).
__device__ __forceinline__ bool is_candidate(const SimGrid& g, V3<double> xi, V3<double> xj, double ri, double rj,
                                             bool outside) {
  double ex = xj.x - xi.x, ey = xj.y - xi.y, ez = xj.z - xi.z;
  if (g.periodic & 1) ex -= product(g.L[0], rint(ex / g.L[0]));
  if (g.periodic & 2) ey -= product(g.L[1], rint(ey / g.L[1]));
  if (g.periodic & 4) ez -= product(g.L[2], rint(ez / g.L[2]));
  const double rs = ri + rj;
  const double d2 = product(ex, ex) + product(ey, ey) + product(ez, ez);
  if (!(d2 < rs * rs * (1.0 + kPrefilterSlack))) return false;
  if (fmax(fabs(ex), fmax(fabs(ey), fabs(ez))) <= g.h * (1.0 - 1e-9) && !outside) return true;
  const double pi[3] = {xi.x, xi.y, xi.z}, pj[3] = {xj.x, xj.y, xj.z};
  uint32_t ci[3], cj[3];
  cell_of(g, pi, ci);
  cell_of(g, pj, cj);
  return cell_slot(g, ci, cj) >= 0;
}

// flag bits of a contact: its neighbour cell's slot in the visit order
__device__ __forceinline__ uint32_t slot_bits(const SimGrid& g, V3<double> xi, V3<double> xj) {
  const double pi[3] = {xi.x, xi.y, xi.z}, pj[3] = {xj.x, xj.y, xj.z};
  uint32_t ci[3], cj[3];
  cell_of(g, pi, ci);
  cell_of(g, pj, cj);
  return (uint32_t)max(cell_slot(g, ci, cj), 0) << kFlagSlot;
}

// Hooke force and torque on the particle at sorted position si of the contact
// ci with the one at sj; the poses' origins in the frame of ci, xi in the world.
template <class T, class R>
__device__ __forceinline__ void contact_force(const DevScene& d, const SimGrid& g, uint32_t si, uint32_t sj,
                                              int32_t matA, int32_t matB, T massA, T massB, V3<double> xi, V3<T> oA,
                                              V3<T> oB, const CInfo<T>& ci, PairRes<R>& out) {
  const HookeP<T> h = hk_table<T>(d)[g.table + material_hash((uint32_t)matA, (uint32_t)matB)];
  const VelRec ri = d.vk[si], rj = d.vk[sj];
  const V3<T> vi = cvt<T>(V3<double>{ri.v[0], ri.v[1], ri.v[2]}), wi = cvt<T>(V3<double>{ri.w[0], ri.w[1], ri.w[2]});
  const V3<T> vj = cvt<T>(V3<double>{rj.v[0], rj.v[1], rj.v[2]}), wj = cvt<T>(V3<double>{rj.w[0], rj.w[1], rj.w[2]});
  V3<T> li, lj;
  if (d.flags & GRAINS_REF_QUIRKS) {
    // reference lever: the world contact point (Kinematics.cpp:86-91)
    V3<T> cpw;
    if constexpr (sizeof(T) == 8)
      cpw = ci.cp;
    else
      cpw = cvt<float>(xi + cvt<double>(ci.cp));
    li = cpw;
    lj = cpw;
  } else {
    li = ci.cp - oA;
    lj = ci.cp - oB;
  }
  const V3<T> relVel = (vi + cross(wi, li)) - (vj + cross(wj, lj));
  const V3<T> relAng = wi - wj;
  V3<T> F, M;
  hooke<T>(h, ci, relVel, relAng, massA, massB, ci.cp - oA, F, M);
  out.f[0] = R(F.x);
  out.f[1] = R(F.y);
  out.f[2] = R(F.z);
  out.m[0] = R(M.x);
  out.m[1] = R(M.y);
  out.m[2] = R(M.z);
}

// Narrow phase + Hooke force of entry (si, sj) -- sorted positions -- from
// si's side (ComponentManagerCPU.cpp:384-419).  Poses come from the sorted
// records; so do velocities, needed only for contacts.  Returns the pair flag.
// e: the entry.  FILTER: apply the prefilter first (a list entry); the
// returned flag is 0 for a pair it leaves out.
// dir (FP32, physics semantics; may be null): receives the direction the
// search ended on in the world frame (left alone when GJK did not run).
// PAIR (physics semantics): lanes 2k and 2k + 1 evaluate
// the same entry, sharing GJK's support pairs (gjk_sv<PAIR>).
// BALLS: every particle is a sphere.
template <class T, class R, bool SV, bool WARM = false, bool PAIR = false, bool FILTER = false, bool BALLS = false>
__device__ __forceinline__ uint32_t pair_force(const DevScene& d, uint32_t si, uint32_t sj, PairRes<R>& out,
                                               NpStats& st, uint32_t e, V3<T>* dir = nullptr) {
  const uint64_t n = d.n;
  const PoseRec pi = d.pk[si];
  const PoseRec pj = d.pk[sj];
  const SimGrid& g = d.grids[pi.sim];
  if constexpr (FILTER) {
    if (!is_candidate(g, V3<double>{pi.x, pi.y, pi.z}, V3<double>{pj.x, pj.y, pj.z}, d.rcs[si], d.rcs[sj],
                      d.nl[kNlOutside] != 0))
      return 0u;
  }
  const ShapeNP<T>* np = np_table<T>(d);
  const ShapeNP<T> A = np[pi.shape];
  const ShapeNP<T> B = np[pj.shape];
  const V3<double> xi = {pi.x, pi.y, pi.z};
  Tr<T> a2w, b2w;
  pair_frames<T>(g, xi, Qt<double>{pi.qx, pi.qy, pi.qz, pi.qw}, V3<double>{pj.x, pj.y, pj.z},
                 Qt<double>{pj.qx, pj.qy, pj.qz, pj.qw}, a2w, b2w);
  // the FP64 re-run of FP32-mixed entries searches to the FP64 path's
  // tolerance, so it decides as that path does
  const GjkArgs args = {d.flags, sizeof(T) == 8 && d.precision == GRAINS_FP32_MIXED ? d.gjk_rel64 : d.gjk_rel};
  CInfo<T> ci;
  if constexpr (BALLS) {
    ci = cp_spheres(A.rc, B.rc, a2w, b2w);
  } else if constexpr (sizeof(T) == 4 && SV && WARM) {
    float4* rec = d.ws + (uint64_t)(*d.ws_par) * ((uint64_t)d.K * n) + e;
    V3<T> dw = {T(0), T(0), T(0)};
    ci = closest_points<T, SV, PAIR>(A, B, a2w, b2w, args, vt_full<T>(d), vt_core<T>(d), st, WarmLookup{rec},
                                             &dw);
    // every entry writes its record (a zero direction when GJK did not run),
    // so none holds the direction of an earlier step
    *rec = make_float4(dw.x, dw.y, dw.z, __uint_as_float(d.sidx[sj]));
    if (dir) *dir = dw;
  } else {
    ci = closest_points<T, SV, PAIR>(A, B, a2w, b2w, args, vt_full<T>(d), vt_core<T>(d), st, NoWarm(), dir);
  }
  uint32_t flag = kFlagCand | (st.gjk() ? kFlagGjk : 0u) | (st.deep() ? kFlagDeep : 0u);
  if (ci.overlap < T(0)) {
    flag |= kFlagContact | slot_bits(g, xi, V3<double>{pj.x, pj.y, pj.z});
    contact_force<T, R>(d, g, si, sj, A.material, B.material, A.mass, B.mass, xi, a2w.o, b2w.o, ci,
                        out);
  }
  return flag;
}

// The step's first kernel, block 0: latch whether the step runs (the lists
// hold) and whether it is the run's last, and clear the integration's queues.
__device__ __forceinline__ bool step_begin(const DevScene& d) {
  const bool run = d.nl[kNlValid] != 0u;
  if (blockIdx.x == 0 && threadIdx.x == 0) {
    d.nl[kNlRun] = run ? 1u : 0u;
    d.nl[kNlLast] = d.nl[kNlDone] + 1u == d.nl[kNlTarget] ? 1u : 0u;
    d.obs_count[0] = d.obs_count[1] = d.obs_count[2] = 0u;  // [1]: pend_count, [2]: obs_count2
  }
  return run;
}
// The last kernel of the step that every step launches once, one thread: the
// step is taken; the narrow phase's queues (no kernel reads them any more).
__device__ __forceinline__ void step_end(const DevScene& d) {
  if (blockIdx.x || threadIdx.x) return;
  d.nl[kNlDone] += 1u;
  d.nl[kNlStale] = d.nl[kNlLast] || d.keep_torce || !d.skin ? 0u : 1u;
  if (d.nl[kNlValid] == 2u) d.nl[kNlValid] = 0u;  // lists for one step
  *d.refine_count = 0u;
  *d.queue_next = 0u;
#pragma unroll
  for (uint32_t q = 0; q < kDeferQueues; ++q) d.defer_count[16 * q] = 0u;
}

// The screen's undecided entries: collected per wave in LDS, appended to the
// block's queue 64 or more at a time and at the end.  Called by whole waves;
// cnt is wave-uniform.
struct DeferLds {
  uint32_t buf[kBlock / 64][128];
  uint32_t cnt[kBlock / 64];
  uint32_t base;
};
__device__ __forceinline__ void defer_push(const DevScene& d, DeferLds& L, uint32_t& cnt, bool pred, uint32_t e) {
  const uint64_t m = __ballot(pred);
  if (!m) return;
  const uint32_t lane = __lane_id(), wv = threadIdx.x / 64;
  if (pred) L.buf[wv][cnt + (uint32_t)__popcll(m & ((1ull << lane) - 1ull))] = e;
  cnt += (uint32_t)__popcll(m);
  if (cnt < 64) return;
  __builtin_amdgcn_fence(__ATOMIC_SEQ_CST, "workgroup");  // the wave's LDS writes are done
  const uint32_t q = blockIdx.x % kDeferQueues;
  uint32_t base = 0;
  if (lane == 0) base = atomicAdd(&d.defer_count[16 * q], cnt);
  base = __shfl(base, 0);
  uint32_t* list = d.defer_list + (uint64_t)q * d.defer_cap + base;
  for (uint32_t k = lane; k < cnt; k += 64) list[k] = L.buf[wv][k];
  __builtin_amdgcn_fence(__ATOMIC_SEQ_CST, "workgroup");  // read before the buffer is refilled
  cnt = 0;
}
__device__ __forceinline__ void defer_flush(const DevScene& d, DeferLds& L, uint32_t cnt) {  // the whole block
  const uint32_t lane = __lane_id(), wv = threadIdx.x / 64, nw = blockDim.x / 64;
  if (lane == 0) L.cnt[wv] = cnt;
  __syncthreads();
  uint32_t off = 0, tot = 0;
  for (uint32_t w = 0; w < nw; ++w) {
    if (w < wv) off += L.cnt[w];
    tot += L.cnt[w];
  }
  const uint32_t q = blockIdx.x % kDeferQueues;
  if (threadIdx.x == 0 && tot) L.base = atomicAdd(&d.defer_count[16 * q], tot);
  __syncthreads();
  if (!tot) return;
  uint32_t* list = d.defer_list + (uint64_t)q * d.defer_cap + L.base + off;
  for (uint32_t k = lane; k < cnt; k += 64) list[k] = L.buf[wv][k];
}

// One lane per list entry, grid-stride.  SV: physics semantics (signed-volume
// GJK); !SV: REF_QUIRKS.
// PASS 0 (the step's only pass): every list entry, complete.  PASS 1: the
// entries that a pass before it queued -- the screen, which settles most, or in
// FP64 the filter, which leaves out those beyond the prefilter -- packed
// lane-dense, complete.  A wave costs as much as its slowest lane, so the long
// searches are kept together and the first pass's waves stay short.  The
// queued searches start from scratch with the same arithmetic: results equal
// those of a single pass bit for bit.
// WARM: FP32 searches start from the pair's previous direction (d.warm).
// PAIR (PASS 1): two lanes per queued entry, sharing its
// support evaluations (pair_force<PAIR>): the queue is short on beds, and
// the pass lasts as long as its longest search (k_complete chooses).
// BALLS (PASS 0, FP64): every particle is a sphere -- no search, no second pass.
// PACK (PASS 0): a wave takes 64 entries at a time that pass the prefilter
// from the list, which holds the skin's too, a quarter to a half as many again
// (FP32 from cold, 40,000 touching superquadrics, ms a step with lists built
// for every step, entries where they stand, packed: 0.986, 1.055, 0.913;
// the reference semantics: kPackNarrow).
template <class T, bool SV, int PASS, bool WARM = false, bool PAIR = false, bool BALLS = false, bool PACK = false>
__device__ __forceinline__ void narrow(const DevScene& d) {
  constexpr bool first = PASS != 1;  // the step's first kernel
  if constexpr (first) {
    if (!step_begin(d)) return;
  }
  PairRes<T>* res = (PairRes<T>*)d.pair_res;
  const uint32_t E = PASS == 1 ? defer_total(d) : d.entry_off[d.n];
  constexpr uint32_t L2 = PAIR ? 2u : 1u;  // lanes per entry
  uint32_t c_cand = 0, c_gjk = 0, c_it = 0, c_deep = 0, c_ref = 0, c_bk = 0, c_maxit = 0, c_near = 0;
  const uint64_t gid = (uint64_t)blockIdx.x * blockDim.x + threadIdx.x;
  const uint64_t stride = (uint64_t)gridDim.x * blockDim.x / L2;
  const bool lead = gid % L2 == 0;  // the lane that stores the entry's results
  const uint32_t lane = __lane_id();
  auto turn = [&](uint32_t e, bool in) {  // an entry per lane (or pair of lanes), whole waves
    uint32_t flag = 0;
    NpStats st = {0u, 0};
    bool refine = false;
    if (in) {
      PairRes<T> r;
      V3<T> dir = {T(0), T(0), T(0)};
      flag = pair_force<T, T, SV, WARM, PAIR, first && !PACK, BALLS>(d, d.pair_i[e], d.pair_j[e], r, st, e,
                                                            sizeof(T) == 4 && SV ? &dir : nullptr);
      if constexpr (first) c_cand += (flag & kFlagCand) != 0;
      // FP32-mixed: re-run in FP64 when the search ended on rounding instead
      // of the gap test, the cores overlap (the contact normal switches to the
      // centre line there), the contact decision lay within FP32's rounding
      // band (its FP64 decision may differ), or (GRAINS_FP64_CONTACTS) the
      // pair is in contact
      refine = sizeof(T) == 4 &&
               (st.backup() || st.deep() || st.near() ||
                ((d.flags & GRAINS_FP64_CONTACTS) && (flag & kFlagContact)));
      if (lead) {
        if (refine) {
          // the FP64 re-run replaces this entry's result: its slot carries the
          // direction the FP32 search ended on, the re-run's first direction
          if (d.res64) {
            PairRes<double> q = {{(double)dir.x, (double)dir.y, (double)dir.z}, {0.0, 0.0, 0.0}};
            ((PairRes<double>*)d.pair_res)[e] = q;
          } else {
            PairRes<T> q;
            q.f[0] = dir.x, q.f[1] = dir.y, q.f[2] = dir.z;
            q.m[0] = q.m[1] = q.m[2] = T(0);
            res[e] = q;
          }
          flag |= kFlagRefine;
        } else if (flag & kFlagContact) {
          // (FP32-mixed with FP64 contact geometry refines every contact)
          res[e] = r;
        }
        d.pair_flag[e] = flag;
        c_gjk += st.gjk();
        c_it += st.iters;
        c_maxit = c_maxit > (uint32_t)st.iters ? c_maxit : (uint32_t)st.iters;
        c_deep += st.deep();
        c_bk += st.backup();
        c_ref += refine;
        c_near += st.near();
      }
    }
    if constexpr (sizeof(T) == 4) wave_append(d.refine_list, d.refine_count, refine && lead, e);
  };
  // whole waves take turns (the queue appends are wave-wide)
  if constexpr (PACK) {
    __shared__ uint32_t packed[kBlock / 64][128];
    uint32_t* mine = packed[threadIdx.x / 64];
    uint32_t have = 0;  // the wave's entries in it
    const bool outside = d.nl[kNlOutside] != 0;
    // a share of the list dealt to each wave, the rest in turn (FP32, physics
    // semantics: most entries end at once) or handed out through a counter (the
    // first queue's: no pass queues entries here)
    constexpr bool turns = sizeof(T) == 4 && SV;
    const uint64_t dealt = stride / 64;
    const uint32_t share =
        64u * (turns ? 1u : (uint32_t)min((uint64_t)8, max((uint64_t)1, (uint64_t)E / (dealt * 64 * 8))));
    uint64_t kw = (gid / 64) * share, end = min((uint64_t)E, kw + share);
    bool more = dealt * share < E;
    for (;;) {
      while (have < 64) {
        if (kw >= end) {
          if (!more) break;
          if constexpr (turns) {
            kw += stride - 64;
          } else {
            uint32_t next = 0;
            if (lane == 0) next = atomicAdd(d.defer_count, share);
            kw = dealt * share + __shfl(next, 0);
          }
          end = min((uint64_t)E, kw + share);
          more = end < E;
          if (kw >= end) break;
        }
        const uint32_t e = (uint32_t)kw + lane;
        bool cand = false;
        if (kw + lane < end) {
          const uint32_t si = d.pair_i[e], sj = d.pair_j[e];
          const PoseRec pi = d.pk[si], pj = d.pk[sj];
          cand = is_candidate(d.grids[pi.sim], V3<double>{pi.x, pi.y, pi.z}, V3<double>{pj.x, pj.y, pj.z}, d.rcs[si],
                              d.rcs[sj], outside);
          if (!cand) {
            if constexpr (WARM) {
              // a pair that left the prefilter's reach forgets its direction
              if (d.pair_flag[e] & kFlagCand)
                d.ws[(uint64_t)(*d.ws_par) * ((uint64_t)d.K * d.n) + e] =
                    make_float4(0.f, 0.f, 0.f, __uint_as_float(d.sidx[sj]));
            }
            d.pair_flag[e] = 0u;
          }
        }
        const uint64_t m = __ballot(cand);
        if (cand) mine[have + (uint32_t)__popcll(m & ((1ull << lane) - 1ull))] = e;
        have += (uint32_t)__popcll(m);
        kw += 64;
      }
      if (!have) break;
      __builtin_amdgcn_fence(__ATOMIC_SEQ_CST, "workgroup");  // the wave's LDS writes are done
      const bool in = lane < have;
      turn(in ? mine[lane] : 0u, in);
      have -= min(have, 64u);
      const uint32_t rest = lane < have ? mine[64 + lane] : 0u;
      __builtin_amdgcn_fence(__ATOMIC_SEQ_CST, "workgroup");  // read before the list is refilled
      if (lane < have) mine[lane] = rest;
    }
  } else {
    for (uint64_t kw = (gid - lane) / L2; kw < E; kw += stride) {
      const uint64_t k = kw + lane / L2;
      const bool in = k < E;
      turn(!in ? 0u : (PASS == 1 ? defer_entry(d, (uint32_t)k) : (uint32_t)k), in);
    }
  }
  if constexpr (first) count_add(d.counters, kCntCandidates, c_cand);
  count_add(d.counters, kCntGjk, c_gjk);
  count_add(d.counters, kCntGjkIters, c_it);
  count_add(d.counters, kCntDeep, c_deep);
  count_add(d.counters, kCntRefine, c_ref);
  count_add(d.counters, kCntBackup, c_bk);
  count_add(d.counters, kCntNear, c_near);
  count_max(d.counters, kCntMaxIters, c_maxit);
}

// One pass, but FP64 under the physics semantics.  The reference's: a list taken as it stands costs as
// many waves as it is long, the skin's entries among them: on large beds more
// than the lists' builds it saves, so those pack it, with as many waves as are
// resident at once; small beds have lanes to spare, and spheres no search.
// Boxes and superquadrics, ms a step with lists built for every step, kept and
// unpacked, packed: FP32 5,000 grains 0.363, 0.238, 0.244, 20,000 0.463, 0.390,
// 0.377, 150,000 1.055, 1.065, 0.927, 500,000 2.77, 2.94, 2.68; FP64 5,000
// 0.348, 0.265, 0.282, 20,000 0.578, 0.596, 0.480, 150,000 2.44, 2.87, 2.12.
constexpr uint64_t kPackNarrow = 10000;  // the largest bed whose list is taken as it stands
template <class T, bool PACK, bool SV = false, bool WARM = false>
__global__ void __launch_bounds__(kBlock) k_narrow(DevScene d) {
  narrow<T, SV, 0, WARM, false, false, PACK>(d);
}
template <class T>
inline void launch_narrow_ref(const DevScene& d, hipStream_t s) {
  if (d.balls || d.n <= kPackNarrow)
    hipLaunchKernelGGL((k_narrow<T, false>), dim3(d.narrow_blocks), dim3(d.block), 0, s, d);
  else
    hipLaunchKernelGGL((k_narrow<T, true>), dim3(std::min(d.narrow_blocks, (unsigned)(cu_count() * kBlock) / d.block)),
                       dim3(d.block), 0, s, d);
}

// Beds of spheres in FP64 (either semantics) take one small pass: screen and
// search passes 6.6 + 13 us on 1,000 spheres, this 7.2 us.
template <class T>
__global__ void __launch_bounds__(kBlock) k_narrow_balls(DevScene d) {
  narrow<T, true, 0, false, false, true>(d);
}

// the screen's part of a shape, in registers from here on
template <class T>
__device__ __forceinline__ void load_now(ShapeNP<T>& s) {
  asm volatile("" : "+v"(s.kind), "+v"(s.rc), "+v"(s.crust), "+v"(s.bbox[0]), "+v"(s.bbox[1]), "+v"(s.bbox[2]));
  asm volatile("" : "+v"(s.core[0]), "+v"(s.core[1]), "+v"(s.core[2]), "+v"(s.core[3]), "+v"(s.core[4]));
}

// The screening pass: screen_pair (REF_QUIRKS: screen_ref) on every entry; the
// entries it leaves undecided go to the complete pass's queues.
// What it costs is waiting for its gathers (a wave of the form that read each
// piece where it was used waited nine loads in turn, 74 % of its time) and,
// behind that, some 700 VALU instructions per entry.  So what is stored by
// entry is read a turn ahead, the shapes at once with what the tests need of
// them, the grid through the scalar cache and a neighbour's id not at all
// (the record keeps it): three waits in turn.  4.2e6 entries of 10^6
// superquadrics: 180 -> 142 us; 128 VGPRs, four waves per SIMD (at 96 it
// spills).  The dies' shares halve what is read past the L2s (710 -> 408 MB).
template <class T, bool WARM, bool SV = true>
__global__ void __launch_bounds__(kBlock, sizeof(T) == 4 ? 4 : 2) k_screen(DevScene d) {
  if (!step_begin(d)) return;
  __shared__ DeferLds L;
  uint32_t nq = 0;  // the wave's entries in L.buf
  const uint32_t E = d.entry_off[d.n], lane = __lane_id();
  float4* const ws = WARM ? d.ws + (uint64_t)(*d.ws_par) * ((uint64_t)d.K * d.n) : nullptr;
  const bool outside = d.nl[kNlOutside] != 0;
  // each die takes a share of the entries (neighbours meet in its L2), its
  // blocks in turn
  const uint32_t dies = gridDim.x % kXcds == 0 ? kXcds : 1;
  const uint32_t share = (E / dies / 64 + 1) * 64, x = blockIdx.x % dies;
  const uint32_t end = min(E, (x + 1) * share), turn = gridDim.x / dies * blockDim.x;
  uint32_t c_cand = 0, c_def = 0, c_gjk = 0;
  uint32_t e = x * share + blockIdx.x / dies * blockDim.x + threadIdx.x;
  uint32_t si = 0, sj = 0;
  float4 rec = make_float4(0.f, 0.f, 0.f, 0.f);
  auto fetch = [&](uint32_t k) {  // what is stored by entry, a turn ahead
    if (k >= end) return;
    si = d.pair_i[k];
    sj = d.pair_j[k];
    if constexpr (WARM) rec = ws[k];
  };
  fetch(e);
  // whole waves take turns (the queue appends are wave-wide)
  for (uint32_t ew = e - lane; ew < end; ew += turn, e += turn) {
    const bool in = e < end;
    const uint32_t ci = si, cj = sj;
    const float4 r = rec;
    uint32_t bits = 0;
    V3<float> dw = {0.f, 0.f, 0.f};
    const PoseRec pi = d.pk[ci], pj = d.pk[cj];
    const double ri = d.rcs[ci], rj = d.rcs[cj];
    fetch(e + turn);
    // what the tests read of the shapes, loaded before the first of them
    ShapeNP<T> A = np_table<T>(d)[pi.shape], B = np_table<T>(d)[pj.shape];
    load_now(A);
    load_now(B);
    bool cand = false;
    V3<double> dm;  // from A's centre to B's nearest image
    for (bool done = !in; !done;) {  // one turn per sim among the wave's entries
      const uint32_t sim = __builtin_amdgcn_readfirstlane(pi.sim);
      uint32_t us = sim;
      asm("" : "+s"(us));  // (sim would become the lane's pi.sim where they are equal)
      if (pi.sim == sim) {
        const SimGrid g = uniform_grid(d.grids + us);
        const V3<double> xi = {pi.x, pi.y, pi.z}, xj = {pj.x, pj.y, pj.z};
        cand = is_candidate(g, xi, xj, ri, rj, outside);
        dm = g.periodic ? min_image(g, xj - xi) : xj - xi;
        done = true;
      }
    }
    if (cand) {
      Tr<T> a2w, b2w;
      pair_frames<T>(V3<double>{pi.x, pi.y, pi.z}, Qt<double>{pi.qx, pi.qy, pi.qz, pi.qw}, V3<double>{pj.x, pj.y, pj.z},
                     Qt<double>{pj.qx, pj.qy, pj.qz, pj.qw}, dm, a2w, b2w);
      V3<T> dir = {T(0), T(0), T(0)};
      bits = !SV ? screen_ref<T>(A, B, a2w, b2w) : screen_pair<T>(A, B, a2w, b2w, vt_full<T>(d), vt_core<T>(d), V3<T>{T(r.x), T(r.y), T(r.z)}, dir);
      if constexpr (WARM) {
        // a settled pair keeps the direction of this step or none (the
        // record's fourth word, the neighbour, stays)
        if (!(bits & kNpDeferred)) dw = dir;
      }
    }
    if (in) {
      if (bits & kNpDeferred) {
        d.pend[ci] = d.pend[cj] = 1u;
      } else {
        d.pair_flag[e] = cand ? kFlagCand | (bits & kNpGjk ? kFlagGjk : 0u) : 0u;
        if constexpr (WARM) {
          if (dw.x != 0.f || dw.y != 0.f || dw.z != 0.f || r.x != 0.f || r.y != 0.f || r.z != 0.f)
            ws[e] = make_float4(dw.x, dw.y, dw.z, r.w);
        }
      }
    }
    c_cand += cand;
    c_gjk += (bits & kNpGjk) != 0;
    c_def += (bits & kNpDeferred) != 0;
    defer_push(d, L, nq, (bits & kNpDeferred) != 0, e);
  }
  defer_flush(d, L, nq);
  count_add(d.counters, kCntDeferred, c_def);
  count_add(d.counters, kCntCandidates, c_cand);
  count_add(d.counters, kCntGjk, c_gjk);
}

// The complete pass over the screen's queue: two lanes per entry where the
// launched lanes hold the queue twice over, else one.  (One launch: the two
// forms as launches of their own cost a graph node of ~5 us each, and the one
// with nothing to do had to wait for room beside the integration: 0.13 ms on
// the bed of 10^6.)  FP32 in 256 threads, 131,072 lanes, ms by two lanes and
// by one: 11,000 entries 0.109 and 0.123, 28,000 0.111 and 0.118, 63,000 0.124
// and 0.119; past the lanes two take another turn: 80,000 0.199 and 0.129,
// 173,000 0.318 and 0.212, 262,000 0.425 and 0.289.
// REF_QUIRKS in FP64 takes the two passes too: in one pass a wave searched
// with the fifth of its lanes that reach GJK.  4,001 boxes and superquadrics
// 149 -> 8 + 93 us.
template <class T, bool WARM, bool SV = true>
__global__ void __launch_bounds__(kBlock) k_complete(DevScene d) {
  // (the FP64 filter's queue may be long: two lanes while they are resident at
  // once, a wave per SIMD.  ms a step by one and by two: 1,000 touching
  // superquadrics, 7,900 entries, 0.71 and 0.48; 3,001 cylinders and cones,
  // 41,000, 0.31 and 0.42)
  constexpr uint64_t resident = sizeof(T) == 8 && SV ? 65536 : ~0ull;
  if ((uint64_t)defer_total(d) * 2 <= min((uint64_t)gridDim.x * blockDim.x, resident))
    narrow<T, SV, 1, WARM, true>(d);
  else
    narrow<T, SV, 1, WARM, false>(d);
}

// Particle x obstacle of any other kind than Rectangle: closestPointsRigidBodies
// (bounding spheres, OBB, GJK) against the obstacle at rest, with its zero
// kinematics and mass (ComponentManagerCPU.cpp:301-351), in FP64 for both
// precisions (obstacle contacts are few; no FP32 re-run is needed).
__device__ __forceinline__ void obstacle_contact64(const DevScene& d, uint32_t si, uint32_t os, const double* t,
                                                   uint32_t table, V3<double> xi, Qt<double> qi, V3<double> vel,
                                                   V3<double> om, V3<double>& F, V3<double>& M, uint32_t& walls,
                                                   NpStats& st) {
  const ShapeNP<double> A = d.np64[si];
  const ShapeNP<double> B = d.np64[os];
  Tr<double> a2w, b2w;
  a2w.R = rot(qi);
  a2w.o = xi;
#pragma unroll
  for (int k = 0; k < 9; ++k) b2w.R.m[k] = t[k];
  b2w.o = {t[9], t[10], t[11]};
  // the FP32-mixed path searches obstacles to its FP64 tolerance
  const GjkArgs args = {d.flags, d.precision == GRAINS_FP32_MIXED ? d.gjk_rel64 : d.gjk_rel};
  const bool quirks = (d.flags & GRAINS_REF_QUIRKS) != 0;
  const CInfo<double> ci =
      quirks ? closest_points<double, false>(A, B, a2w, b2w, args, d.verts64, d.cverts64, st)
             : closest_points<double, true>(A, B, a2w, b2w, args, d.verts64, d.cverts64, st);
  if (ci.overlap < 0.0) {
    const HookeP<double> h = d.hooke64[table + material_hash((uint32_t)A.material, (uint32_t)B.material)];
    const V3<double> lever = quirks ? ci.cp : ci.cp - xi;
    const V3<double> relVel = vel + cross(om, lever);
    V3<double> f, m;
    hooke<double>(h, ci, relVel, om, A.mass, B.mass, ci.cp - xi, f, m);
    F = F + f;
    M = M + m;
    ++walls;
  }
}

// Particle x Rectangle wall at rest: the plane branch of
// closestPointsRigidBodies (CollisionDetection.cpp:203-206) and the Hooke
// force f and torque m, in FP64; returns whether they touch.  Walls whose plane is
// farther from the centre than every point of the particle leave the support
// point on its side: no contact, decided without it.
template <bool BALLS = false>
__device__ __forceinline__ bool wall_contact64(const DevScene& d, const ShapeNP<double>& A0, uint32_t o,
                                               uint32_t table, V3<double> xi, Qt<double> qi, V3<double> vel,
                                               V3<double> om, V3<double>& f, V3<double>& m) {
  ShapeNP<double> A = A0;
  if (BALLS) A.kind = GRAINS_SPHERE;
  const double* t = d.obs_tr + 12 * (size_t)o;
  const uint32_t os = d.obs_shape[o];
  Tr<double> a2w, b2w;
#pragma unroll
  for (int k = 0; k < 9; ++k) b2w.R.m[k] = t[k];
  b2w.o = {t[9], t[10], t[11]};
  const V3<double> rn = {t[2], t[5], t[8]};
  if (fabs(dot(rn, xi - b2w.o)) > A.rc_max * (1.0 + 1e-9)) return false;
  a2w.R = rot(qi);
  a2w.o = xi;
  const CInfo<double> ci = cp_rectangle(sup_ctx(A, false, d.verts64, d.cverts64), a2w, b2w);
  if (!(ci.overlap < 0.0)) return false;
  const ShapeNP<double> B = d.np64[os];
  const HookeP<double> h = d.hooke64[table + material_hash((uint32_t)A.material, (uint32_t)B.material)];
  // reference lever: the world contact point (Kinematics.cpp:86-91)
  const V3<double> lever = (d.flags & GRAINS_REF_QUIRKS) ? ci.cp : ci.cp - a2w.o;
  const V3<double> relVel = vel + cross(om, lever);
  hooke<double>(h, ci, relVel, om, A.mass, B.mass, ci.cp - a2w.o, f, m);
  return true;
}

// Can particle i (centre xi, every point within rc_max of it) touch an
// obstacle of its sim?  Rectangles: the centre's distance from the plane;
// other kinds: the two bounding spheres (closestPointsRigidBodies tests them
// first).  Conservative by 1e-9 relative, so a particle it clears is one the
// full test finds out of contact.
__device__ __forceinline__ bool obstacle_in_reach(const DevScene& d, const SimGrid& g, double rc_max,
                                                  V3<double> xi) {
  for (uint32_t o = g.obs_begin; o < g.obs_end; ++o) {
    const double* t = d.obs_tr + 12 * (size_t)o;
    const V3<double> xo = {t[9], t[10], t[11]};
    const ShapeNP<double>& B = d.np64[d.obs_shape[o]];
    const double reach = B.kind == GRAINS_RECTANGLE ? fabs(dot(V3<double>{t[2], t[5], t[8]}, xi - xo))
                                                    : norm(xi - xo) - B.rc_max;
    if (reach <= rc_max * (1.0 + 1e-9)) return true;
  }
  return false;
}

struct IntegCounts {
  uint32_t walls = 0, contacts = 0, gjk = 0, iters = 0, deep = 0, nonfinite = 0, outside = 0, max_cand = 0;
  __device__ __forceinline__ void add(const IntegCounts& c) {
    walls += c.walls;
    contacts += c.contacts;
    gjk += c.gjk;
    iters += c.iters;
    deep += c.deep;
    nonfinite += c.nonfinite;
    outside += c.outside;
    max_cand = max(max_cand, c.max_cand);
  }
};

// The contacts of sorted position s, summed in the reference's visit order.
// The list stands in the visit order of the positions it was built from;
// particles that have changed cell since can leave contacts out of order, and
// then the sum is taken again in order (two contacts sum the same either way).
template <class T>
__device__ __forceinline__ void sum_contacts(const DevScene& d, uint32_t s, V3<double>& F, V3<double>& M,
                                             int32_t& ncon, uint32_t& ncand) {
  const PairRes<T>* res = (const PairRes<T>*)d.pair_res;
  const PairRes<double>* res64 = (const PairRes<double>*)d.pair_res;  // d.res64
  const uint32_t e0 = d.entry_off[s], e1 = d.entry_off[s + 1];
  F = M = {0.0, 0.0, 0.0};
  ncon = 0;
  ncand = 0;
  auto add = [&](uint32_t e) {
    if (sizeof(T) == 4 && d.res64) {
      const PairRes<double> r = res64[e];
      F = F + V3<double>{r.f[0], r.f[1], r.f[2]};
      M = M + V3<double>{r.m[0], r.m[1], r.m[2]};
    } else {
      const PairRes<T> r = res[e];
      F = F + V3<double>{(double)r.f[0], (double)r.f[1], (double)r.f[2]};
      M = M + V3<double>{(double)r.m[0], (double)r.m[1], (double)r.m[2]};
    }
  };
  auto order = [&](uint32_t fl, uint32_t e) {  // (slot, id) in the visit order
    return ((uint64_t)((fl >> kFlagSlot) & 31u) << 32) | d.sidx[d.pair_j[e]];
  };
  bool sorted = true;
  uint32_t last_fl = 0, last_e = 0;
  // four flags loaded together (one load latency per four)
  for (uint32_t e = e0; e < e1; e += 4) {
    uint32_t fl[4];
#pragma unroll
    for (uint32_t u = 0; u < 4; ++u) fl[u] = e + u < e1 ? d.pair_flag[e + u] : 0u;
#pragma unroll
    for (uint32_t u = 0; u < 4; ++u) {
      ncand += (fl[u] & kFlagCand) != 0;
      if (fl[u] & kFlagContact) {
        add(e + u);
        if (ncon) {
          const uint32_t a = last_fl >> kFlagSlot, b = fl[u] >> kFlagSlot;
          sorted &= a < b || (a == b && order(last_fl, last_e) < order(fl[u], e + u));
        }
        last_fl = fl[u];
        last_e = e + u;
        ++ncon;
      }
    }
  }
  if (!sorted && ncon > 2) {
    F = M = {0.0, 0.0, 0.0};
    uint64_t done = 0;
    for (int32_t k = 0; k < ncon; ++k) {
      uint64_t best = ~0ull;
      uint32_t be = e0;
      for (uint32_t e = e0; e < e1; ++e) {
        const uint32_t fl = d.pair_flag[e];
        if (!(fl & kFlagContact)) continue;
        const uint64_t o = order(fl, e);
        if ((k == 0 || o > done) && o < best) best = o, be = e;
      }
      add(be);
      done = best;
    }
  }
}

// The state at the step's start of the particle at sorted position s.
struct ParticleState {
  uint32_t si, sim;
  V3<double> xi, vel, om;
  Qt<double> qi;
  __device__ __forceinline__ ParticleState(const DevScene& d, uint32_t s) {
    const PoseRec p = d.pk[s];
    const VelRec v = d.vk[s];
    si = p.shape, sim = p.sim;
    xi = {p.x, p.y, p.z};
    qi = {p.qx, p.qy, p.qz, p.qw};
    vel = {v.v[0], v.v[1], v.v[2]};
    om = {v.w[0], v.w[1], v.w[2]};
  }
};

// Gravity, then moveParticles (ComponentManagerCPU.cpp:428-500) on the
// quaternion state, from the total contact force F and torque M.  SO: a
// second-order scheme (d.integrator); otherwise FirstOrderExplicit.
template <bool SO>
__device__ __forceinline__ void finish_step(const DevScene& d, const SimGrid& g, uint32_t s, const ParticleState& p0,
                                            V3<double> F, V3<double> M, int32_t ncon, uint32_t ncand,
                                            IntegCounts& c) {
  const uint64_t n = d.n;
  const uint32_t si = p0.si;
  const V3<double> xi = p0.xi, vel = p0.vel, om = p0.om;
  const Qt<double> qi = p0.qi;
  // addExternalForces (ComponentManagerCPU.cpp:448-460)
  const Dynamics dy = load_dyn(d.dyn + si);
  F = F + dy.mass * V3<double>{g.g[0], g.g[1], g.g[2]};
  c.contacts = (uint32_t)ncon;
  c.max_cand = ncand;
  c.outside = xi.x < g.lo[0] || xi.x > g.hi[0] || xi.y < g.lo[1] || xi.y > g.hi[1] || xi.z < g.lo[2] || xi.z > g.hi[2];
  const bool asked = d.nl[kNlLast] || d.keep_torce;  // the results of the run's last step can be asked for
  const uint64_t i = asked || ncon || !d.skin ? d.sidx[s] : 0u;
  if (ncon) d.contact_count[i] += ncon;
  if (asked) {
    store3(d.last_force, n, i, F);
    store3(d.last_torque, n, i, M);
    // the reference's cell of the step's positions
    const double p[3] = {xi.x, xi.y, xi.z};
    uint32_t cc[3];
    cell_of(g, p, cc);
    d.key[i] = cell_key(g, cc);
  }
  V3<double> x = xi, vnew = vel, onew = om;
  Qt<double> qn = qi;
  if constexpr (!SO) {
    move_particle(dy.mass, dy.inertia, dy.inv, d.dt, F, M, x, qn, vnew, onew);
  } else {
    V3<double> hist[4];
    const int nh = d.integrator == GRAINS_SECOND_ORDER_ADAMS_BASHFORTH ? 4
                   : d.integrator == GRAINS_SECOND_ORDER_LEAPFROG    ? 1
                                                                     : 0;
    double* h = d.hk + 12 * (uint64_t)s;
    for (int k = 0; k < nh; ++k) hist[k] = {h[3 * k], h[3 * k + 1], h[3 * k + 2]};
    move_particle_scheme(d.integrator, dy.mass, dy.inertia, dy.inv, d.dt, F, M, x, qn, vnew, onew, hist);
    for (int k = 0; k < nh; ++k) h[3 * k] = hist[k].x, h[3 * k + 1] = hist[k].y, h[3 * k + 2] = hist[k].z;
  }
  if (g.periodic) {
    // periodic wrap of the centre (not in the reference)
    auto wrap = [&](double cc, int k) {
      if (!((g.periodic >> k) & 1)) return cc;
      if (cc < g.lo[k]) return cc + g.L[k];
      if (cc >= g.hi[k]) return cc - g.L[k];
      return cc;
    };
    x = {wrap(x.x, 0), wrap(x.y, 1), wrap(x.z, 2)};
  }
  // the pose record in list order; the lists hold while every particle is
  // within half the skin of where they were built, inside its periodic sides
  PoseRec pr;
  pr.x = x.x, pr.y = x.y, pr.z = x.z;
  pr.qx = qn.x, pr.qy = qn.y, pr.qz = qn.z, pr.qw = qn.w;
  pr.shape = si;
  pr.sim = p0.sim;
  const VelRec vr = {{vnew.x, vnew.y, vnew.z}, {onew.x, onew.y, onew.z}};
  d.pk[s] = pr;
  d.vk[s] = vr;
  if (d.skin) {
    const double4 b = d.bp[s];
    V3<double> mv = {x.x - b.x, x.y - b.y, x.z - b.z};
    if (g.periodic) mv = min_image(g, mv);
    bool out = mv.x * mv.x + mv.y * mv.y + mv.z * mv.z > g.move2;
    if (g.periodic) {
      const double p[3] = {x.x, x.y, x.z};
#pragma unroll
      for (int k = 0; k < 3; ++k) out |= ((g.periodic >> k) & 1) && (p[k] < g.lo[k] || p[k] >= g.hi[k]);
    }
    if (out) d.nl[kNlValid] = 0u;
  }
  // the planes, when they are read before another build (step_end tells it)
  if (asked || !d.skin) store_state(d, i, s, pr, vr);
  // a non-finite state (NaN or infinity anywhere in it) is counted; the
  // reference has no such check and carries NaN on silently
  const double all = x.x + x.y + x.z + qn.x + qn.y + qn.z + qn.w + vnew.x + vnew.y + vnew.z + onew.x + onew.y + onew.z;
  c.nonfinite = !isfinite(all);
}

// One particle's step from its sorted position s: its contacts, obstacles
// (one lane takes them in turn, some not Rectangles; FP64 for both
// precisions; ComponentManagerCPU.cpp:301-351), gravity and the move.
template <class T, bool SO>
__device__ __forceinline__ void integrate_obs(const DevScene& d, uint32_t s, IntegCounts& c) {
  V3<double> F, M;
  int32_t ncon;
  uint32_t ncand;
  sum_contacts<T>(d, s, F, M, ncon, ncand);
  const ParticleState p(d, s);
  const SimGrid& g = d.grids[p.sim];
  const ShapeNP<double> A = d.np64[p.si];
  for (uint32_t o = g.obs_begin; o < g.obs_end; ++o) {
    const uint32_t os = d.obs_shape[o];
    if (d.np64[os].kind != GRAINS_RECTANGLE) {
      NpStats st = {0u, 0};
      obstacle_contact64(d, p.si, os, d.obs_tr + 12 * (size_t)o, g.table, p.xi, p.qi, p.vel, p.om, F, M, c.walls, st);
      c.gjk += st.gjk();
      c.iters += st.iters;
      c.deep += st.deep();
    } else {
      V3<double> f, m;
      if (wall_contact64(d, A, o, g.table, p.xi, p.qi, p.vel, p.om, f, m)) {
        F = F + f;
        M = M + m;
        ++c.walls;
      }
    }
  }
  finish_step<SO>(d, g, s, p, F, M, ncon, ncand, c);
}

__device__ __forceinline__ void integrate_counts(const DevScene& d, const IntegCounts& c, bool gen) {
  count_add(d.counters, kCntNan, c.nonfinite);
  count_add(d.counters, kCntWall, c.walls);
  // contacts are counted after any FP64 re-run has settled each entry
  count_add(d.counters, kCntContacts, c.contacts);
  count_add(d.counters, kCntOod, c.outside);
  count_max(d.counters, kCntMaxCand, c.max_cand);
  if (gen) {
    count_add(d.counters, kCntGjk, c.gjk);
    count_add(d.counters, kCntGjkIters, c.iters);
    count_add(d.counters, kCntDeep, c.deep);
  }
}

// One particle (sorted position s) without obstacle contacts, or its queueing
// for k_integrate_obs; returns whether it was queued.
template <class T, bool SO>
__device__ __forceinline__ bool integrate_or_queue(const DevScene& d, const SimGrid& g, uint32_t s,
                                                   const ParticleState& p, double reach, IntegCounts& c) {
  if (g.obs_end > g.obs_begin && obstacle_in_reach(d, g, reach, p.xi)) return true;
  V3<double> F, M;
  int32_t ncon;
  uint32_t ncand;
  sum_contacts<T>(d, s, F, M, ncon, ncand);
  finish_step<SO>(d, g, s, p, F, M, ncon, ncand, c);
  return false;
}

// One thread per particle, in list order.  A particle within reach of an obstacle of its
// sim is queued for k_integrate_obs instead (obs_list); the others need no
// obstacle code, so this kernel does not carry the FP64 support maps and
// GJK that obstacle contacts take.  SPLIT: a particle the screen marked
// (d.pend) is queued in pend_list for k_integrate_pend instead.
// Bound by what it moves, ~360 B a particle from and to its records in list
// order; one thread per particle id, with the state in planes, the pose
// record scattered beside them and 176 B of shape read for one radius, moved
// 684 B and took 154 us for 10^6 superquadrics (beside the complete pass);
// now 105 us.
template <class T, bool SO, bool SPLIT = false>
__global__ void __launch_bounds__(kBlock) k_integrate(DevScene d) {
  if (!d.nl[kNlRun]) return;
  if (!SPLIT) step_end(d);
  const uint64_t s = (uint64_t)blockIdx.x * blockDim.x + threadIdx.x;
  IntegCounts c;
  bool queue = false, later = false;
  if (s < d.n) {
    const bool marked = d.pend[s] != 0u;
    if (!SPLIT && marked) d.pend[s] = 0u;
    later = SPLIT && marked;
    if (!later) {
      const ParticleState p(d, (uint32_t)s);
      const double reach = d.nobs ? d.rws[s] : 0.0;
      for (bool done = false; !done;) {  // one turn per sim among the wave's particles
        const uint32_t sim = __builtin_amdgcn_readfirstlane(p.sim);
        uint32_t us = sim;
        asm("" : "+s"(us));  // (sim would become the lane's p.sim where they are equal)
        if (p.sim == sim) {
          queue = integrate_or_queue<T, SO>(d, uniform_grid(d.grids + us), (uint32_t)s, p, reach, c);
          done = true;
        }
      }
    }
  }
  if (SPLIT) wave_append(d.pend_list, d.pend_count, later, (uint32_t)s);
  if (d.nobs) wave_append(d.obs_list, d.obs_count, queue, (uint32_t)s);
  integrate_counts(d, c, false);
}

// The particles k_integrate<SPLIT> queued in pend_list, as k_integrate.
// Block-strided over the queue, whose length the device holds; every lane of
// a wave takes the same number of turns (the queue appends are wave-wide).
template <class T, bool SO>
__global__ void __launch_bounds__(kBlock) k_integrate_pend(DevScene d) {
  if (!d.nl[kNlRun]) return;
  step_end(d);
  const uint32_t cnt = *d.pend_count;
  IntegCounts tot;
  const uint64_t stride = (uint64_t)gridDim.x * blockDim.x;
  for (uint64_t b = (uint64_t)blockIdx.x * blockDim.x; b < cnt; b += stride) {
    const uint64_t k = b + threadIdx.x;
    bool queue = false;
    uint32_t s = 0;
    if (k < cnt) {
      s = d.pend_list[k];
      d.pend[s] = 0u;
      IntegCounts c;
      // (a queued wave holds particles of many sims)
      const ParticleState p(d, s);
      queue = integrate_or_queue<T, SO>(d, d.grids[p.sim], s, p, d.nobs ? d.rws[s] : 0.0, c);
      tot.add(c);
    }
    if (d.nobs) wave_append(d.obs_list2, d.obs_count2, queue, s);
  }
  integrate_counts(d, tot, false);
}

// The particles k_integrate (list obs_list) or k_integrate_pend (obs_list2)
// queued: the same step with their obstacle contacts (FP64; some obstacles
// are not Rectangles).  Grid-stride over the queue, whose length the device
// holds.
template <class T, bool SO>
__global__ void __launch_bounds__(kBlock) k_integrate_obs(DevScene d, const uint32_t* __restrict__ list,
                                                         const uint32_t* __restrict__ count) {
  if (!d.nl[kNlRun]) return;
  const uint32_t cnt = *count;
  IntegCounts tot;
  const uint64_t stride = (uint64_t)gridDim.x * blockDim.x;
  for (uint64_t k = (uint64_t)blockIdx.x * blockDim.x + threadIdx.x; k < cnt; k += stride) {
    IntegCounts c;
    integrate_obs<T, SO>(d, list[k], c);
    tot.add(c);
  }
  integrate_counts(d, tot, true);
}

// The same where every obstacle is a Rectangle, by eight lanes per particle:
// each takes one wall (a superquadric's support is a chain of seven FP64 pow
// calls: one lane taking a corner grain's walls in turn held its wave ~25 us),
// and the contacts are added in the walls' order.
// ALL: every particle instead of a queue -- a small bed's whole integration
// in one launch, the step's last (1,000 spheres: 16 + 25 us in two launches -> 18 us;
// 8,191 touching superquadrics: 22 + 90 us -> 27 us).
template <class T, bool SO, bool ALL, bool BALLS = false>
__global__ void __launch_bounds__(kBlock) k_integrate_walls(DevScene d, const uint32_t* __restrict__ list,
                                                           const uint32_t* __restrict__ count) {
  if (!d.nl[kNlRun]) return;
  if (ALL) step_end(d);
  constexpr uint32_t G = 8;
  const uint32_t cnt = ALL ? (uint32_t)d.n : *count;
  const uint32_t lane = __lane_id(), sub = lane % G;
  IntegCounts tot;
  const uint64_t stride = (uint64_t)gridDim.x * blockDim.x / G;
  for (uint64_t k = ((uint64_t)blockIdx.x * blockDim.x + threadIdx.x) / G; k < cnt; k += stride) {
    const uint32_t s = ALL ? (uint32_t)k : list[k];
    const ParticleState p(d, s);
    const SimGrid& g = d.grids[p.sim];
    V3<double> F, M;
    int32_t ncon;
    uint32_t ncand;
    sum_contacts<T>(d, s, F, M, ncon, ncand);
    uint32_t walls = 0;
    for (uint32_t o0 = g.obs_begin; o0 < g.obs_end; o0 += G) {
      V3<double> f = {0.0, 0.0, 0.0}, m = f;
      const bool hit = o0 + sub < g.obs_end &&
                       wall_contact64<BALLS>(d, d.np64[p.si], o0 + sub, g.table, p.xi, p.qi, p.vel, p.om, f, m);
      uint32_t hits = (uint32_t)(__ballot(hit) >> (lane - sub)) & ((1u << G) - 1u);
      for (; hits; hits &= hits - 1) {
        const int w = (int)(lane - sub) + __ffs(hits) - 1;
        F = F + V3<double>{__shfl(f.x, w), __shfl(f.y, w), __shfl(f.z, w)};
        M = M + V3<double>{__shfl(m.x, w), __shfl(m.y, w), __shfl(m.z, w)};
        ++walls;
      }
    }
    if (sub == 0) {
      if (ALL && d.pend[s]) d.pend[s] = 0u;
      IntegCounts c;
      c.walls = walls;
      finish_step<SO>(d, g, s, p, F, M, ncon, ncand, c);
      tot.add(c);
    }
  }
  integrate_counts(d, tot, false);
}

// The integration launches of one precision (launch_integrate32/64).
// part 1 (second stream): the particles the screen settled, then their
// obstacle queue; part 2 (after the join): the marked particles, then
// theirs; part 0: every particle (a bed of at most kWideIntegrate by eight
// lanes each where all obstacles are Rectangles), then the obstacle queue.
template <class T, bool SO>
inline void launch_integrate_so(const DevScene& d, hipStream_t s, int part) {
  const dim3 grid((unsigned)((d.n + d.block - 1) / d.block)), block(d.block);
  // queues are walked grid-stride over their device-held counts
  const dim3 og(std::min<unsigned>(grid.x, (unsigned)cu_count() * 8));
  if (part == 0 && d.nobs && !d.gen_obs && d.n <= kWideIntegrate) {
    const dim3 eight((unsigned)((d.n * 8 + kBlock - 1) / kBlock));
    if (sizeof(T) == 8 && d.balls)
      hipLaunchKernelGGL((k_integrate_walls<T, SO, true, sizeof(T) == 8>), eight, dim3(kBlock), 0, s, d, nullptr, nullptr);
    else
      hipLaunchKernelGGL((k_integrate_walls<T, SO, true>), eight, dim3(kBlock), 0, s, d, nullptr, nullptr);
    return;
  }
  if (part == 1)
    hipLaunchKernelGGL((k_integrate<T, SO, true>), grid, block, 0, s, d);
  else if (part == 2)
    hipLaunchKernelGGL((k_integrate_pend<T, SO>), og, block, 0, s, d);
  else
    hipLaunchKernelGGL((k_integrate<T, SO>), grid, block, 0, s, d);
  if (!d.nobs) return;
  const uint32_t* list = part == 2 ? d.obs_list2 : d.obs_list;
  const uint32_t* count = part == 2 ? d.obs_count2 : d.obs_count;
  if (d.gen_obs)
    hipLaunchKernelGGL((k_integrate_obs<T, SO>), og, block, 0, s, d, list, count);
  else
    hipLaunchKernelGGL((k_integrate_walls<T, SO, false>), dim3((unsigned)cu_count() * 2), dim3(kBlock), 0, s, d, list,
                       count);
}
template <class T>
inline void launch_integrate_t(const DevScene& d, hipStream_t s, int part) {
  if (d.integrator != GRAINS_FIRST_ORDER_EXPLICIT)
    launch_integrate_so<T, true>(d, s, part);
  else
    launch_integrate_so<T, false>(d, s, part);
}

// GrainsTestDev workload: GJK distance of independent pairs of full shapes.
template <class T, bool SV>
__device__ __forceinline__ void gjk_batch(const ShapeNP<T>* shapes, const T* verts, const uint32_t* __restrict__ sa,
                                          const uint32_t* __restrict__ sb, const double* __restrict__ ta,
                                          const double* __restrict__ tb, uint64_t n, const GjkArgs& args,
                                          double* __restrict__ dist, double* __restrict__ pa,
                                          double* __restrict__ pb, int32_t* __restrict__ iters) {
  const uint64_t k = (uint64_t)blockIdx.x * blockDim.x + threadIdx.x;
  if (k >= n) return;
  const double* A12 = ta + 12 * k;
  const double* B12 = tb + 12 * k;
  Tr<T> a2w, b2w;
#pragma unroll
  for (int c = 0; c < 9; ++c) {
    a2w.R.m[c] = T(A12[c]);
    b2w.R.m[c] = T(B12[c]);
  }
  const V3<double> xa = {A12[9], A12[10], A12[11]}, xb = {B12[9], B12[10], B12[11]};
  if constexpr (sizeof(T) == 8) {
    a2w.o = xa;
    b2w.o = xb;
  } else {
    a2w.o = {0.0f, 0.0f, 0.0f};
    b2w.o = cvt<float>(xb - xa);
  }
  const ShapeNP<T> A = shapes[sa[k]], B = shapes[sb[k]];
  SupCtx<T> ca = sup_ctx(A, false, verts, verts);
  SupCtx<T> cb = sup_ctx(B, false, verts, verts);
  GjkOut<T> g;
  if constexpr (SV)
    g = gjk_sv(ca, cb, a2w, b2w, args, A.rc + B.rc, T(INFINITY));
  else
    g = gjk_jh(ca, cb, a2w, b2w, args);
  dist[k] = (double)g.dist;
  if (iters) iters[k] = g.iters;
  if (pa) {
    V3<double> p = cvt<double>(apply(a2w, g.pa)), q = cvt<double>(apply(b2w, g.pb));
    if constexpr (sizeof(T) == 4) {
      p = p + xa;
      q = q + xa;
    }
    pa[3 * k] = p.x;
    pa[3 * k + 1] = p.y;
    pa[3 * k + 2] = p.z;
    pb[3 * k] = q.x;
    pb[3 * k + 1] = q.y;
    pb[3 * k + 2] = q.z;
  }
}

template <class T, bool SV>
__global__ void __launch_bounds__(kBlock) k_gjk_batch(const ShapeNP<T>* __restrict__ shapes,
                                                     const T* __restrict__ verts, const uint32_t* __restrict__ sa,
                                                     const uint32_t* __restrict__ sb, const double* __restrict__ ta,
                                                     const double* __restrict__ tb, uint64_t n, GjkArgs args,
                                                     double* __restrict__ dist, double* __restrict__ pa,
                                                     double* __restrict__ pb, int32_t* __restrict__ iters) {
  gjk_batch<T, SV>(shapes, verts, sa, sb, ta, tb, n, args, dist, pa, pb, iters);
}
// A few shapes without vertices ride in the kernel's arguments instead of
// memory allocated, filled and freed around the launch (614,400 pairs in FP32:
// 215 -> 125 us; the witness points it does not return leave it 168
// registers instead of 241, three waves per SIMD).
template <class T>
struct ArgShapes {
  ShapeNP<T> s[kArgShapes];
};
template <class T, bool SV>
__global__ void __launch_bounds__(kBlock, sizeof(T) == 4 && !SV ? 3 : 1) k_gjk_batch_args(ArgShapes<T> shapes, const uint32_t* __restrict__ sa,
                                                          const uint32_t* __restrict__ sb,
                                                          const double* __restrict__ ta,
                                                          const double* __restrict__ tb, uint64_t n, GjkArgs args,
                                                          double* __restrict__ dist, int32_t* __restrict__ iters) {
  gjk_batch<T, SV>(shapes.s, nullptr, sa, sb, ta, tb, n, args, dist, nullptr, nullptr, iters);
}
template <class T>
inline void launch_gjk_batch_args_t(const ShapeNP<T>* shapes, size_t count, const uint32_t* sa, const uint32_t* sb,
                                    const double* ta, const double* tb, uint64_t n, GjkArgs args, double* dist,
                                    int32_t* iters, hipStream_t s) {
  ArgShapes<T> a{};
  std::copy(shapes, shapes + count, a.s);
  const dim3 grid((unsigned)((n + 63) / 64)), block(64);  // a wave's registers are free when it ends
  if (args.flags & GRAINS_REF_QUIRKS)
    hipLaunchKernelGGL((k_gjk_batch_args<T, false>), grid, block, 0, s, a, sa, sb, ta, tb, n, args, dist, iters);
  else
    hipLaunchKernelGGL((k_gjk_batch_args<T, true>), grid, block, 0, s, a, sa, sb, ta, tb, n, args, dist, iters);
}

}  // namespace gr
