// gr_narrow.hpp -- per-entry narrow phase + contact force, per-particle
// reduction + walls + gravity + explicit integration, and the standalone GJK
// batch.  Included by gr_narrow64.hip (T = double, built without FMA
// contraction) and gr_narrow32.hip (T = float, FP32-mixed).
#pragma once

#include <algorithm>

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

// The previous step's GJK direction of the pair (wi, wj), looked up only
// when the pair reaches GJK: wi's entry wk of the previous step first (a
// particle's list keeps its order while its neighbours stay), then its other
// entries, four loads in flight at a time.  Records: float4 {direction in the
// world frame, neighbour id bits} in entry order; nb = {first entry, count}
// of wi in the previous step.
struct WarmLookup {
  const float4* prev;
  const uint2* prev_nb;
  uint32_t wi, wj, wk;
  GR_D bool fetch(V3<float>& w) const {
    const uint2 nb = prev_nb[wi];
    const uint32_t np = nb.y;
    const float4* pr = prev + nb.x;
    float4 r = make_float4(0.f, 0.f, 0.f, 0.f);
    bool hit = false;
    if (wk < np) {
      r = pr[wk];
      hit = __float_as_uint(r.w) == wj;
    }
    for (uint32_t k0 = 0; !hit && k0 < np; k0 += 4) {
      float4 q[4];
#pragma unroll
      for (uint32_t u = 0; u < 4; ++u)
        q[u] = k0 + u < np ? pr[k0 + u] : make_float4(0.f, 0.f, 0.f, 0.f);
#pragma unroll
      for (uint32_t u = 0; u < 4; ++u)
        if (!hit && k0 + u < np && __float_as_uint(q[u].w) == wj) {
          r = q[u];
          hit = true;
        }
    }
    w = {r.x, r.y, r.z};
    const float nn = dot(w, w);
    return hit && nn > 0.f && nn < INFINITY;
  }
};

// Hooke force and torque on particle i of the contact ci with j; the poses'
// origins in the frame of ci, xi in the world.
template <class T, class R>
__device__ __forceinline__ void contact_force(const DevScene& d, const SimGrid& g, uint32_t i, uint32_t j,
                                              int32_t matA, int32_t matB, T massA, T massB, V3<double> xi, V3<T> oA,
                                              V3<T> oB, const CInfo<T>& ci, PairRes<R>& out) {
  const uint64_t n = d.n;
  const HookeP<T> h = hk_table<T>(d)[g.table + material_hash((uint32_t)matA, (uint32_t)matB)];
  const V3<T> vi = cvt<T>(load3(d.vel, n, i)), wi = cvt<T>(load3(d.omega, n, i));
  const V3<T> vj = cvt<T>(load3(d.vel, n, j)), wj = cvt<T>(load3(d.omega, n, j));
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
// records; velocities, needed only for contacts, from the planes through the
// particle ids.  Returns the pair flag.
// e: the entry (its slot in si's candidate list keys the warm-start record);
// ~0u for callers without one (the FP64 re-run).
// dir (FP32, physics semantics; may be null): receives the direction the
// search ended on in the world frame (left alone when GJK did not run).
// PAIR (physics semantics): lanes 2k and 2k + 1 evaluate
// the same entry, sharing GJK's support pairs (gjk_sv<PAIR>).
template <class T, class R, bool SV, bool SCREEN = false, bool WARM = false, bool PAIR = false>
__device__ __forceinline__ uint32_t pair_force(const DevScene& d, uint32_t si, uint32_t sj, PairRes<R>& out,
                                               NpStats& st, uint32_t e = ~0u, V3<T>* dir = nullptr) {
  const uint64_t n = d.n;
  const PoseRec pi = d.pk[si];
  const PoseRec pj = d.pk[sj];
  const ShapeNP<T>* np = np_table<T>(d);
  const ShapeNP<T> A = np[pi.shape];
  const ShapeNP<T> B = np[pj.shape];
  const SimGrid& g = d.grids[pi.sim];
  const V3<double> xi = {pi.x, pi.y, pi.z};
  Tr<T> a2w, b2w;
  pair_frames<T>(g, xi, Qt<double>{pi.qx, pi.qy, pi.qz, pi.qw}, V3<double>{pj.x, pj.y, pj.z},
                 Qt<double>{pj.qx, pj.qy, pj.qz, pj.qw}, a2w, b2w);
  // the FP64 re-run of FP32-mixed entries searches to the FP64 path's
  // tolerance, so it decides as that path does
  const GjkArgs args = {d.flags, sizeof(T) == 8 && d.precision == GRAINS_FP32_MIXED ? d.gjk_rel64 : d.gjk_rel};
  CInfo<T> ci;
  if constexpr (sizeof(T) == 4 && SV && WARM) {
    if (e != ~0u) {
      const uint64_t KN = (uint64_t)d.K * n;
      const uint32_t cur = *d.ws_par;
      const uint32_t wj = d.sidx[sj];
      const WarmLookup wl{d.ws + (uint64_t)(1u - cur) * KN, d.ws_nb + (uint64_t)(1u - cur) * n, d.sidx[si], wj,
                          e - d.entry_off[si]};
      V3<T> dw = {T(0), T(0), T(0)};
      ci = closest_points<T, SV, SCREEN, PAIR>(A, B, a2w, b2w, args, vt_full<T>(d), vt_core<T>(d), st, wl, &dw);
      // every decided entry writes its record (a zero direction when GJK
      // did not run), so an entry never holds a record of an earlier step
      if (!st.deferred()) d.ws[(uint64_t)cur * KN + e] = make_float4(dw.x, dw.y, dw.z, __uint_as_float(wj));
      if (dir) *dir = dw;
    } else {
      ci = closest_points<T, SV, SCREEN, PAIR>(A, B, a2w, b2w, args, vt_full<T>(d), vt_core<T>(d), st, NoWarm(),
                                               dir);
    }
  } else {
    ci = closest_points<T, SV, SCREEN, PAIR>(A, B, a2w, b2w, args, vt_full<T>(d), vt_core<T>(d), st, NoWarm(), dir);
  }
  uint32_t flag = (st.gjk() ? kFlagGjk : 0u) | (st.deep() ? kFlagDeep : 0u);
  if constexpr (SCREEN) return flag;  // decided pairs have no contact
  if (ci.overlap < T(0)) {
    flag |= kFlagContact;
    contact_force<T, R>(d, g, d.sidx[si], d.sidx[sj], A.material, B.material, A.mass, B.mass, xi, a2w.o, b2w.o, ci,
                        out);
  }
  return flag;
}

// One lane per candidate entry, grid-stride.  SV: physics semantics
// (signed-volume GJK); !SV: REF_QUIRKS.
// PASS 0: every entry, complete.  With two passes (physics semantics):
// PASS 2 screens every entry -- bounding sphere, OBB and GJK's first support
// pair decide most pairs of a resting or loose packing (no contact) with a
// small kernel -- and queues the rest; PASS 1 runs the queued entries, packed
// lane-dense, complete.  A wave costs as much as its slowest lane, so the
// long searches are kept together and the screen's waves stay short.  The
// queued searches start from scratch with the same arithmetic: results equal
// those of PASS 0 bit for bit.
// The screen queues into one segment per block (an LDS counter, no global
// atomic: a single queue counter would serialise one atomic per wave); the
// segments are copied into one list at the offsets of an exclusive scan of
// their counts (launch_defer_flatten), which PASS 1 reads in order.
// WARM: FP32 searches start from the pair's previous direction (d.warm).
// PAIR (PASS 1, physics semantics): two lanes per queued entry, sharing its
// support evaluations (pair_force<PAIR>): the queue is short on beds, and
// the pass lasts as long as its longest search.  The PAIR launch runs when
// the grid holds the queue twice over, the other when it does not (each
// returns at once in the other's case).
template <class T, bool SV, int PASS, bool WARM = false, bool PAIR = false>
__global__ void __launch_bounds__(kBlock) k_narrow(DevScene d) {
  constexpr bool screen = SV && PASS == 2;
  __shared__ uint32_t seg_n;
  uint32_t* seg = d.defer_list + (uint64_t)blockIdx.x * d.defer_cap;
  if constexpr (screen) {
    if (threadIdx.x == 0) seg_n = 0;
    __syncthreads();
  }
  PairRes<T>* res = (PairRes<T>*)d.pair_res;
  const uint32_t E = PASS == 1 ? d.defer_off[gridDim.x] : d.entry_off[d.n];
  if constexpr (PASS == 1) {
    const bool paired = SV && (uint64_t)E * 2 <= (uint64_t)gridDim.x * blockDim.x;
    if (paired != PAIR) return;
  }
  constexpr uint32_t L = PAIR ? 2u : 1u;  // lanes per entry
  uint32_t c_gjk = 0, c_it = 0, c_deep = 0, c_ref = 0, c_bk = 0, c_maxit = 0, c_near = 0;
  const uint64_t gid = (uint64_t)blockIdx.x * blockDim.x + threadIdx.x;
  const uint64_t stride = (uint64_t)gridDim.x * blockDim.x / L;
  const bool lead = gid % L == 0;  // the lane that stores the entry's results
  for (uint64_t k = gid / L; k < E; k += stride) {
    uint32_t e = (uint32_t)k;
    if constexpr (PASS == 1) e = d.defer_flat[k];
    NpStats st = {0u, 0};
    PairRes<T> r;
    V3<T> dir = {T(0), T(0), T(0)};
    uint32_t flag = pair_force<T, T, SV, screen, WARM, PAIR>(d, d.pair_i[e], d.pair_j[e], r, st, e,
                                                              sizeof(T) == 4 && SV ? &dir : nullptr);
    if constexpr (screen) {
      block_append(seg, &seg_n, st.deferred() != 0, e);
      if (st.deferred()) d.pend[d.pair_i[e]] = d.pend[d.pair_j[e]] = 1u;
    }
    // FP32-mixed: re-run in FP64 when the search ended on rounding instead
    // of the gap test, the cores overlap (the contact normal switches to the
    // centre line there), the contact decision lay within FP32's rounding
    // band (its FP64 decision may differ), or (GRAINS_FP64_CONTACTS) the
    // pair is in contact
    const bool refine = sizeof(T) == 4 && !st.deferred() &&
                        (st.backup() || st.deep() || st.near() ||
                         ((d.flags & GRAINS_FP64_CONTACTS) && (flag & kFlagContact)));
    if (!st.deferred() && lead) {
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
    if constexpr (sizeof(T) == 4 && !screen) wave_append(d.refine_list, d.refine_count, refine && lead, e);
  }
  if constexpr (screen) {
    __syncthreads();
    if (threadIdx.x == 0) d.defer_count[blockIdx.x] = seg_n;
    count_add(d.counters, kCntDeferred, threadIdx.x == 0 ? seg_n : 0u);  // every lane: a wave reduction
  }
  count_add(d.counters, kCntGjk, c_gjk);
  count_add(d.counters, kCntGjkIters, c_it);
  count_add(d.counters, kCntDeep, c_deep);
  count_add(d.counters, kCntRefine, c_ref);
  count_add(d.counters, kCntBackup, c_bk);
  count_add(d.counters, kCntNear, c_near);
  count_max(d.counters, kCntMaxIters, c_maxit);
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
// force, in FP64; adds to F and M and returns 1 on contact.
__device__ __forceinline__ uint32_t wall_contact64(const DevScene& d, const ShapeNP<double>& A, uint32_t os,
                                                   uint32_t table, const Tr<double>& a2w, const Tr<double>& b2w,
                                                   V3<double> vel, V3<double> om, V3<double>& F, V3<double>& M) {
  const CInfo<double> ci = cp_rectangle(sup_ctx(A, false, d.verts64, d.cverts64), a2w, b2w);
  if (!(ci.overlap < 0.0)) return 0;
  const ShapeNP<double> B = d.np64[os];
  const HookeP<double> h = d.hooke64[table + material_hash((uint32_t)A.material, (uint32_t)B.material)];
  // reference lever: the world contact point (Kinematics.cpp:86-91)
  const V3<double> lever = (d.flags & GRAINS_REF_QUIRKS) ? ci.cp : ci.cp - a2w.o;
  const V3<double> relVel = vel + cross(om, lever);
  V3<double> f, m;
  hooke<double>(h, ci, relVel, om, A.mass, B.mass, ci.cp - a2w.o, f, m);
  F = F + f;
  M = M + m;
  return 1;
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
  uint32_t walls = 0, contacts = 0, gjk = 0, iters = 0, deep = 0, nonfinite = 0;
};

// One particle's step from its sorted position s: sum its entries in visit
// order, obstacles (OBS; FP64 for both precisions, GEN: some are not
// Rectangles), gravity, then moveParticles (ComponentManagerCPU.cpp:428-500)
// on the quaternion state.  SO: a second-order scheme (d.integrator);
// otherwise FirstOrderExplicit.
template <class T, bool OBS, bool GEN, bool SO>
__device__ __forceinline__ void integrate_particle(const DevScene& d, uint64_t i, uint32_t s, IntegCounts& c) {
  const uint64_t n = d.n;
  const PairRes<T>* res = (const PairRes<T>*)d.pair_res;
  const PairRes<double>* res64 = (const PairRes<double>*)d.pair_res;  // d.res64
  const uint32_t e0 = d.entry_off[s], e1 = d.entry_off[s + 1];
  V3<double> F = {0.0, 0.0, 0.0}, M = {0.0, 0.0, 0.0};
  int32_t ncon = 0;
  // in entry order; four flags loaded together (one load latency per four)
  for (uint32_t e = e0; e < e1; e += 4) {
    uint32_t fl[4];
#pragma unroll
    for (uint32_t u = 0; u < 4; ++u) fl[u] = e + u < e1 ? d.pair_flag[e + u] : 0u;
#pragma unroll
    for (uint32_t u = 0; u < 4; ++u)
      if (fl[u] & kFlagContact) {
        if (sizeof(T) == 4 && d.res64) {
          const PairRes<double> r = res64[e + u];
          F = F + V3<double>{r.f[0], r.f[1], r.f[2]};
          M = M + V3<double>{r.m[0], r.m[1], r.m[2]};
        } else {
          const PairRes<T> r = res[e + u];
          F = F + V3<double>{(double)r.f[0], (double)r.f[1], (double)r.f[2]};
          M = M + V3<double>{(double)r.m[0], (double)r.m[1], (double)r.m[2]};
        }
        ++ncon;
      }
  }
  const uint32_t si = d.shape[i];
  const SimGrid& g = d.grids[d.sim[i]];
  const V3<double> xi = load3(d.pos, n, i);
  const Qt<double> qi = load_quat(d.quat, n, i);
  const V3<double> vel = load3(d.vel, n, i);
  const V3<double> om = load3(d.omega, n, i);
  // particle x obstacle (ComponentManagerCPU.cpp:301-351)
  if constexpr (OBS) {
    const ShapeNP<double> A = d.np64[si];
    for (uint32_t o = g.obs_begin; o < g.obs_end; ++o) {
      const double* t = d.obs_tr + 12 * (size_t)o;
      const uint32_t os = d.obs_shape[o];
      if constexpr (GEN) {
        if (d.np64[os].kind != GRAINS_RECTANGLE) {
          NpStats st = {0u, 0};
          obstacle_contact64(d, si, os, t, g.table, xi, qi, vel, om, F, M, c.walls, st);
          c.gjk += st.gjk();
          c.iters += st.iters;
          c.deep += st.deep();
          continue;
        }
      }
      Tr<double> a2w, b2w;
#pragma unroll
      for (int k = 0; k < 9; ++k) b2w.R.m[k] = t[k];
      b2w.o = {t[9], t[10], t[11]};
      // a centre farther from the plane than every point of the particle
      // leaves the support point on its side: no contact, decided without it
      const V3<double> rn = {t[2], t[5], t[8]};
      if (fabs(dot(rn, xi - b2w.o)) > A.rc_max * (1.0 + 1e-9)) continue;
      a2w.R = rot(qi);
      a2w.o = xi;
      c.walls += wall_contact64(d, A, os, g.table, a2w, b2w, vel, om, F, M);
    }
  }
  // addExternalForces (ComponentManagerCPU.cpp:448-460)
  const ShapeDyn dy = d.dyn[si];
  F = F + dy.mass * V3<double>{g.g[0], g.g[1], g.g[2]};
  store3(d.last_force, n, i, F);
  store3(d.last_torque, n, i, M);
  d.contact_count[i] += ncon;
  c.contacts = (uint32_t)ncon;
  V3<double> x = xi, vnew = vel, onew = om;
  Qt<double> qn = qi;
  if constexpr (!SO) {
    move_particle(dy.mass, dy.inertia, dy.inv, d.dt, F, M, x, qn, vnew, onew);
  } else {
    V3<double> hist[4];
    const int nh = d.integrator == GRAINS_SECOND_ORDER_ADAMS_BASHFORTH ? 4
                   : d.integrator == GRAINS_SECOND_ORDER_LEAPFROG    ? 1
                                                                     : 0;
    for (int k = 0; k < nh; ++k) hist[k] = load3(d.ab_hist + 3 * k * n, n, i);
    move_particle_scheme(d.integrator, dy.mass, dy.inertia, dy.inv, d.dt, F, M, x, qn, vnew, onew, hist);
    for (int k = 0; k < nh; ++k) store3(d.ab_hist + 3 * k * n, n, i, hist[k]);
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
  store3(d.pos, n, i, x);
  store3(d.vel, n, i, vnew);
  store3(d.omega, n, i, onew);
  d.quat[i] = qn.x;
  d.quat[n + i] = qn.y;
  d.quat[2 * n + i] = qn.z;
  d.quat[3 * n + i] = qn.w;
  // a non-finite state (NaN or infinity anywhere in it) is counted; the
  // reference has no such check and carries NaN on silently
  const double all = x.x + x.y + x.z + qn.x + qn.y + qn.z + qn.w + vnew.x + vnew.y + vnew.z + onew.x + onew.y + onew.z;
  c.nonfinite = !isfinite(all);
}

__device__ __forceinline__ void integrate_counts(const DevScene& d, const IntegCounts& c, bool gen) {
  count_add(d.counters, kCntNan, c.nonfinite);
  count_add(d.counters, kCntWall, c.walls);
  // contacts are counted after any FP64 re-run has settled each entry
  count_add(d.counters, kCntContacts, c.contacts);
  if (gen) {
    count_add(d.counters, kCntGjk, c.gjk);
    count_add(d.counters, kCntGjkIters, c.iters);
    count_add(d.counters, kCntDeep, c.deep);
  }
}

// One particle (id i, sorted position s) without obstacle contacts, or its
// queueing for k_integrate_obs; returns whether it was queued.
template <class T, bool SO>
__device__ __forceinline__ bool integrate_or_queue(const DevScene& d, uint32_t i, uint32_t s, IntegCounts& c) {
  const uint64_t n = d.n;
  if (d.warm) d.ws_nb[(uint64_t)(*d.ws_par) * n + i] = make_uint2(d.entry_off[s], d.entry_off[s + 1] - d.entry_off[s]);
  const SimGrid& g = d.grids[d.sim[i]];
  const bool queue =
      g.obs_end > g.obs_begin && obstacle_in_reach(d, g, d.np64[d.shape[i]].rc_max, load3(d.pos, n, i));
  if (!queue) integrate_particle<T, false, false, SO>(d, i, s, c);
  return queue;
}

// One thread per particle.  A particle within reach of an obstacle of its
// sim is queued for k_integrate_obs instead (obs_list); the others need no
// obstacle code, so this kernel does not carry the FP64 support maps and
// GJK that obstacle contacts take.  SPLIT: a particle the screen marked
// (d.pend) is queued in pend_list for k_integrate_pend instead.
template <class T, bool SO, bool SPLIT = false>
__global__ void __launch_bounds__(kBlock) k_integrate(DevScene d) {
  const uint64_t n = d.n;
  const uint64_t i = (uint64_t)blockIdx.x * blockDim.x + threadIdx.x;
  IntegCounts c;
  bool queue = false, later = false;
  if (i < n) {
    const uint32_t s = d.rank[i];
    later = SPLIT && d.pend[s];
    if (!later) queue = integrate_or_queue<T, SO>(d, (uint32_t)i, s, c);
  }
  if (SPLIT) wave_append(d.pend_list, d.pend_count, later, (uint32_t)i);
  if (d.nobs) wave_append(d.obs_list, d.obs_count, queue, (uint32_t)i);
  integrate_counts(d, c, false);
}

// The particles k_integrate<SPLIT> queued in pend_list, as k_integrate.
// Block-strided over the queue, whose length the device holds; every lane of
// a wave takes the same number of turns (the queue appends are wave-wide).
template <class T, bool SO>
__global__ void __launch_bounds__(kBlock) k_integrate_pend(DevScene d) {
  const uint32_t cnt = *d.pend_count;
  IntegCounts tot;
  const uint64_t stride = (uint64_t)gridDim.x * blockDim.x;
  for (uint64_t b = (uint64_t)blockIdx.x * blockDim.x; b < cnt; b += stride) {
    const uint64_t k = b + threadIdx.x;
    bool queue = false;
    uint32_t i = 0;
    if (k < cnt) {
      i = d.pend_list[k];
      IntegCounts c;
      queue = integrate_or_queue<T, SO>(d, i, d.rank[i], c);
      tot.walls += c.walls;
      tot.contacts += c.contacts;
      tot.nonfinite += c.nonfinite;
    }
    if (d.nobs) wave_append(d.obs_list2, d.obs_count2, queue, i);
  }
  integrate_counts(d, tot, false);
}

// The particles k_integrate (list obs_list) or k_integrate_pend (obs_list2)
// queued: the same step with their obstacle contacts (FP64; GEN: some
// obstacles are not Rectangles).  Grid-stride over the queue, whose length
// the device holds.
template <class T, bool GEN, bool SO>
__global__ void __launch_bounds__(kBlock) k_integrate_obs(DevScene d, const uint32_t* __restrict__ list,
                                                         const uint32_t* __restrict__ count) {
  const uint32_t cnt = *count;
  IntegCounts tot;
  const uint64_t stride = (uint64_t)gridDim.x * blockDim.x;
  for (uint64_t k = (uint64_t)blockIdx.x * blockDim.x + threadIdx.x; k < cnt; k += stride) {
    const uint32_t i = list[k];
    IntegCounts c;
    integrate_particle<T, true, GEN, SO>(d, i, d.rank[i], c);
    tot.walls += c.walls;
    tot.contacts += c.contacts;
    tot.gjk += c.gjk;
    tot.iters += c.iters;
    tot.deep += c.deep;
    tot.nonfinite += c.nonfinite;
  }
  integrate_counts(d, tot, GEN);
}

// The integration launches of one precision (launch_integrate32/64).
// part 1 (second stream): the particles the screen settled, then their
// obstacle queue; part 2 (after the join): the marked particles, then
// theirs; part 0: every particle, then the obstacle queue.
template <class T>
inline void launch_integrate_t(const DevScene& d, hipStream_t s, int part) {
  const dim3 grid((unsigned)((d.n + d.block - 1) / d.block));
  const bool so = d.integrator != GRAINS_FIRST_ORDER_EXPLICIT;
  // queues are walked grid-stride over their device-held counts
  const dim3 og(std::min<unsigned>(grid.x, (unsigned)cu_count() * 8));
  if (part == 1) {
    if (so)
      hipLaunchKernelGGL((k_integrate<T, true, true>), grid, dim3(d.block), 0, s, d);
    else
      hipLaunchKernelGGL((k_integrate<T, false, true>), grid, dim3(d.block), 0, s, d);
  } else if (part == 2) {
    if (so)
      hipLaunchKernelGGL((k_integrate_pend<T, true>), og, dim3(d.block), 0, s, d);
    else
      hipLaunchKernelGGL((k_integrate_pend<T, false>), og, dim3(d.block), 0, s, d);
  } else if (so) {
    hipLaunchKernelGGL((k_integrate<T, true>), grid, dim3(d.block), 0, s, d);
  } else {
    hipLaunchKernelGGL((k_integrate<T, false>), grid, dim3(d.block), 0, s, d);
  }
  if (!d.nobs) return;
  const uint32_t* list = part == 2 ? d.obs_list2 : d.obs_list;
  const uint32_t* count = part == 2 ? d.obs_count2 : d.obs_count;
  if (d.gen_obs && so)
    hipLaunchKernelGGL((k_integrate_obs<T, true, true>), og, dim3(d.block), 0, s, d, list, count);
  else if (d.gen_obs)
    hipLaunchKernelGGL((k_integrate_obs<T, true, false>), og, dim3(d.block), 0, s, d, list, count);
  else if (so)
    hipLaunchKernelGGL((k_integrate_obs<T, false, true>), og, dim3(d.block), 0, s, d, list, count);
  else
    hipLaunchKernelGGL((k_integrate_obs<T, false, false>), og, dim3(d.block), 0, s, d, list, count);
}

// GrainsTestDev workload: GJK distance of independent pairs of full shapes.
template <class T, bool SV>
__global__ void __launch_bounds__(kBlock) k_gjk_batch(const ShapeNP<T>* __restrict__ shapes,
                                                     const T* __restrict__ verts, const uint32_t* __restrict__ sa,
                                                     const uint32_t* __restrict__ sb, const double* __restrict__ ta,
                                                     const double* __restrict__ tb, uint64_t n, GjkArgs args,
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

}  // namespace gr
