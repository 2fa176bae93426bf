// gr_search.hpp -- the FP64 searches of the physics semantics (the complete
// pass of the FP64 path, the FP64 re-runs of the FP32-mixed path): the
// signed-volume GJK of gjk_sv, operation for operation, as a loop over a
// queue of entries in which every turn is one iteration of each lane's own
// search.
#pragma once

#include "gr_narrow.hpp"

namespace gr {

// ---- exchange within a quad of lanes (DPP: no LDS round trip) ----------------------
// CTRL: quad_perm of two bits per lane
template <int CTRL>
__device__ __forceinline__ double quad_get(double x) {
  union {
    double d;
    int i[2];
  } u;
  u.d = x;
  u.i[0] = __builtin_amdgcn_mov_dpp(u.i[0], CTRL, 0xf, 0xf, true);
  u.i[1] = __builtin_amdgcn_mov_dpp(u.i[1], CTRL, 0xf, 0xf, true);
  return u.d;
}
constexpr int kQuadXor1 = 0xB1, kQuadXor2 = 0x4E;              // lanes (1, 0, 3, 2), (2, 3, 0, 1)
constexpr int kQuad0 = 0x00, kQuad1 = 0x55, kQuad2 = 0xAA;     // lane 0, 1, 2 to all four
template <int CTRL>
__device__ __forceinline__ V3<double> quad_get(V3<double> a) {
  return {quad_get<CTRL>(a.x), quad_get<CTRL>(a.y), quad_get<CTRL>(a.z)};
}

// ---- one support, the pow chain of sq_support_pow --------------------------------
// The exponents and ratios come from the shape's SqPow record.  Arguments of
// pow are never negative; saying so (fabs) drops its sign handling.  A
// direction in the plane x = 0 takes the two-dimensional chain through the
// same calls.  SPLIT: the two lanes 2k, 2k + 1 hold the same direction and
// take one each of the two independent calls of a level (five levels instead
// of seven calls).
template <bool SPLIT>
__device__ __forceinline__ void pow2(double x0, double y0, double x1, double y1, double& r0, double& r1) {
  if constexpr (SPLIT) {
    const bool role = (__lane_id() & 1u) != 0;
    const double p = pow(fabs(role ? x1 : x0), role ? y1 : y0);
    const double o = quad_get<kQuadXor1>(p);
    r0 = role ? o : p;
    r1 = role ? p : o;
  } else {
    r0 = pow(fabs(x0), y0);
    r1 = pow(fabs(x1), y1);
  }
}
template <bool SPLIT>
__device__ __forceinline__ V3<double> sq_support_split(const double* d, const SqPow& k, V3<double> v) {
  const double a = d[0], b = d[1], c = d[2], n1 = d[3], n2 = d[4];
  const double ax = fabs(v.x), ay = fabs(v.y), az = fabs(v.z);
  const double sx = sgn(v.x), sy = sgn(v.y), sz = sgn(v.z);
  const bool flat = ax == 0.0;
  if (flat && ay == 0.0) return {0.0, 0.0, sz * c};
  if (n1 == 2.0 && n2 == 2.0) {  // an ellipsoid: every exponent is 1, 0, 2 or 1/2
    const double alpha = (flat ? k.cb : k.ba) * (flat ? az : ay) / (flat ? ay : ax);
    const double beta = k.ca * az / ax;
    const double temp = 1.0 + alpha * alpha;
    const double xt = 1.0 / sqrt(flat ? temp : temp + beta * beta);
    if (flat) return {0.0, sy * b * xt, sz * alpha * c * xt};
    return {sx * a * xt, sy * alpha * b * xt, sz * beta * c * xt};
  }
  double alpha, zeta, gamma, tr;
  pow2<SPLIT>((flat ? k.cb : k.ba) * (flat ? az : ay) / (flat ? ay : ax), flat ? k.k2 : k.k1, k.ca * az / ax,
              k.k2, alpha, zeta);
  const double temp = 1.0 + pow(fabs(alpha), flat ? n1 : n2);
  pow2<SPLIT>(temp, k.g, temp, k.r, gamma, tr);
  const double beta = gamma * zeta;
  const double sum = tr + pow(fabs(beta), n1);
  const double xt = 1.0 / pow(fabs(flat ? temp : sum), k.in1);
  if (flat) return {0.0, sy * b * xt, sz * alpha * c * xt};
  return {sx * a * xt, sy * alpha * b * xt, sz * beta * c * xt};
}

// ---- the simplex ------------------------------------------------------------------
// Closest point of the simplex {y[0], .., y[n-1]} to the origin, newest point
// first: sv_seg / sv_tri / sv_tet with the cases folded, so that the lanes of
// a wave share one triangle and one segment routine whatever their simplex:
// a tetrahedron's faces in turn (usually one), a triangle as its own face, a
// segment as an edge of it.
struct SvBest {
  V3<double> v;
  double lam[4];
  unsigned mask;
};
// (selects, not branches: a branch costs a wave on its own more than the
// segment's arithmetic)
__device__ __forceinline__ void sv_edge(V3<double> a, V3<double> b, V3<double> t, unsigned ib, V3<double>& v,
                                        double& l0, double& l1, unsigned& mask) {
  const double tt = dot(t, t);
  const double l = -dot(a, t) / tt;
  const bool at_b = tt > 0.0 && l >= 1.0, in = tt > 0.0 && l > 0.0 && l < 1.0;
  const V3<double> m = a + l * t;
  v = {in ? m.x : (at_b ? b.x : a.x), in ? m.y : (at_b ? b.y : a.y), in ? m.z : (at_b ? b.z : a.z)};
  l0 = in ? 1.0 - l : (at_b ? 0.0 : 1.0);
  l1 = in ? l : (at_b ? 1.0 : 0.0);
  mask = in ? 1u | (1u << ib) : (at_b ? 1u << ib : 1u);
}
__device__ __forceinline__ SvBest sv_closest(const V3<double>* y, int n) {
  const V3<double> a = y[0];
  SvBest best;
  best.v = a;
  best.lam[0] = 1.0;
  best.lam[1] = best.lam[2] = best.lam[3] = 0.0;
  best.mask = 1u;
  unsigned faces = n == 3 ? 4u : (n == 2 ? 8u : 0u);  // bit f: face without point f + 1 (2: (0, 1, 2)); 8: the edge (0, 1)
  if (n == 4) {
    const V3<double> ab = y[1] - a, ac = y[2] - a, ad = y[3] - a;
    const V3<double> cd = cross(ac, ad);
    const double D = dot(ab, cd);
    double l1 = 0.0, l2 = 0.0, l3 = 0.0;
    bool in = false;
    if (D != 0.0) {
      l1 = -dot(a, cd) / D;
      l2 = dot(ab, cross(ad, a)) / D;
      l3 = dot(ab, cross(a, ac)) / D;
      const double l0 = ((1.0 - l1) - l2) - l3;
      if (l0 > 0.0 && l1 > 0.0 && l2 > 0.0 && l3 > 0.0) {
        in = true;
        best.v = {0.0, 0.0, 0.0};
        best.lam[0] = l0;
        best.lam[1] = l1;
        best.lam[2] = l2;
        best.lam[3] = l3;
        best.mask = 15u;
      }
    }
    if (!in) {
      faces = (D == 0.0 || l1 <= 0.0 ? 1u : 0u) | (D == 0.0 || l2 <= 0.0 ? 2u : 0u) |
              (D == 0.0 || l3 <= 0.0 ? 4u : 0u);
      if (!faces) faces = 7u;
    }
  }
  bool first = true;
  while (faces) {
    const unsigned f = faces & (0u - faces);
    faces ^= f;
    const unsigned ib = f == 1u ? 2u : 1u, ic = f == 4u ? 2u : 3u;
    const V3<double> b = f == 1u ? y[2] : y[1], c = f == 4u ? y[2] : y[3];
    const V3<double> e1 = b - a, e2 = c - a;
    V3<double> v;
    double m0, mb = 0.0, mc = 0.0;
    unsigned mask = 0;
    bool eb = true, ec = false;
    if (f != 8u) {
      const V3<double> nr = cross(e1, e2);
      const double nn = dot(nr, nr);
      double lb = 0.0, lc = 0.0;
      if (nn > 0.0) {
        lb = dot(nr, cross(e2, a)) / nn;
        lc = dot(nr, cross(a, e1)) / nn;
        const double la = (1.0 - lb) - lc;
        if (la > 0.0 && lb > 0.0 && lc > 0.0) {
          v = (a + lb * e1) + lc * e2;
          m0 = la;
          mb = lb;
          mc = lc;
          mask = 1u | (1u << ib) | (1u << ic);
        }
      }
      eb = !(nn > 0.0) || lc <= 0.0;
      ec = !(nn > 0.0) || lb <= 0.0;
      if (!eb && !ec) eb = ec = true;  // only a's weight is not positive (rounding): keep a's edges
    }
    if (!mask) {
      const unsigned i1 = eb ? ib : ic;
      double s0, s1;
      sv_edge(a, eb ? b : c, eb ? e1 : e2, i1, v, s0, s1, mask);
      m0 = s0;
      mb = eb ? s1 : 0.0;
      mc = eb ? 0.0 : s1;
      if (eb && ec) {
        V3<double> u;
        unsigned um;
        sv_edge(a, c, e2, ic, u, s0, s1, um);
        if (norm2(u) < norm2(v)) {
          v = u;
          m0 = s0;
          mb = 0.0;
          mc = s1;
          mask = um;
        }
      }
    }
    if (first || norm2(v) < norm2(best.v)) {
      best.v = v;
      best.mask = mask;
      best.lam[0] = m0;
      best.lam[1] = ib == 1u ? mb : 0.0;
      best.lam[2] = ib == 2u ? mb : (ic == 2u ? mc : 0.0);
      best.lam[3] = ic == 3u ? mc : 0.0;
    }
    first = false;
  }
  return best;
}

// First vertex of the largest v.x (support's POLYHEDRON case), the vertices
// shared by the two lanes of a body: one takes the even, the other the odd
// ones, four loads in flight, and the larger value wins, the lower index
// among equals.
__device__ __forceinline__ V3<double> poly_support_split(const double* P, int nv, V3<double> v) {
  const int role = (int)(__lane_id() & 1u);
  V3<double> best = {P[0], P[1], P[2]};
  double bd = dot(v, best);
  int bi = 0;
  for (int i0 = role; i0 < nv; i0 += 8) {
    V3<double> p[4];
#pragma unroll
    for (int u = 0; u < 4; ++u) {
      const int i = i0 + 2 * u < nv ? i0 + 2 * u : 0;
      p[u] = {P[3 * i], P[3 * i + 1], P[3 * i + 2]};
    }
#pragma unroll
    for (int u = 0; u < 4; ++u) {
      const double dd = dot(v, p[u]);
      if (i0 + 2 * u < nv && dd > bd) {
        bd = dd;
        best = p[u];
        bi = i0 + 2 * u;
      }
    }
  }
  const double od = quad_get<kQuadXor1>(bd);
  const int oi = __builtin_amdgcn_mov_dpp(bi, kQuadXor1, 0xf, 0xf, true);
  const V3<double> ob = quad_get<kQuadXor1>(best);
  const bool take = od > bd || (od == bd && oi < bi);
  return {take ? ob.x : best.x, take ? ob.y : best.y, take ? ob.z : best.z};
}

// sv_closest by the four lanes of a quad, each holding its face: a
// tetrahedron's three coordinates, then its three faces, one per lane, then
// the best of the faces that count, in their order.  A search on its own in a
// wave is a chain of dependent FP64 instructions (~10 cycles each); the faces
// one after another were most of it for shapes without pow.
// b, c: the older points of the lane's face (lane 0: points 2 and 3, 1: 1 and
// 3, 2 and 3: 1 and 2; a: the newest, point 0).
__device__ __forceinline__ SvBest sv_closest_quad(V3<double> a, V3<double> b, V3<double> c, int n) {
  const uint32_t q = __lane_id() & 3u;
  SvBest best;
  unsigned faces = 4u;
  double l1 = 0.0, l2 = 0.0, l3 = 0.0, l0 = 0.0;
  bool in = false;
  const V3<double> e1 = b - a, e2 = c - a;
  if (n == 4) {
    // lane 0: u = ac x ad, 1: ad x a, 2: a x ac
    const V3<double> X = {q == 2 ? a.x : (q == 1 ? e2.x : e1.x), q == 2 ? a.y : (q == 1 ? e2.y : e1.y),
                          q == 2 ? a.z : (q == 1 ? e2.z : e1.z)};
    const V3<double> Y = {q == 1 ? a.x : e2.x, q == 1 ? a.y : e2.y, q == 1 ? a.z : e2.z};
    const V3<double> ab = quad_get<kQuad1>(e1);
    const V3<double> u = cross(X, Y);
    const double D = quad_get<kQuad0>(dot(ab, u));
    const V3<double> Z = {q == 0 ? a.x : ab.x, q == 0 ? a.y : ab.y, q == 0 ? a.z : ab.z};
    const double num = dot(Z, u);
    const double l = (q == 0 ? -num : num) / D;
    l1 = quad_get<kQuad0>(l);
    l2 = quad_get<kQuad1>(l);
    l3 = quad_get<kQuad2>(l);
    l0 = ((1.0 - l1) - l2) - l3;
    in = D != 0.0 && l0 > 0.0 && l1 > 0.0 && l2 > 0.0 && l3 > 0.0;
    faces = (D == 0.0 || l1 <= 0.0 ? 1u : 0u) | (D == 0.0 || l2 <= 0.0 ? 2u : 0u) | (D == 0.0 || l3 <= 0.0 ? 4u : 0u);
    if (!faces) faces = 7u;
  }
  // the lane's face; a segment: its edge (0, 1) only
  const V3<double> nr = cross(e1, e2);
  const double nn = dot(nr, nr);
  const bool tri = n >= 3 && nn > 0.0;
  const double lb = tri ? dot(nr, cross(e2, a)) / nn : 0.0;
  const double lc = tri ? dot(nr, cross(a, e1)) / nn : 0.0;
  const double la = (1.0 - lb) - lc;
  const bool inner = tri && la > 0.0 && lb > 0.0 && lc > 0.0;
  bool eb = !tri || lc <= 0.0, ec = n >= 3 && (!tri || lb <= 0.0);
  if (n >= 3 && !eb && !ec) eb = ec = true;  // only a's weight is not positive (rounding): keep a's edges
  V3<double> vb, vc;
  double b0, b1, c0, c1;
  unsigned kb, kc;
  sv_edge(a, b, e1, 1u, vb, b0, b1, kb);
  sv_edge(a, c, e2, 2u, vc, c0, c1, kc);
  const bool useb = eb && !(ec && norm2(vc) < norm2(vb));
  const V3<double> vi = (a + lb * e1) + lc * e2;
  const bool pt = n == 1;
  V3<double> v = {inner ? vi.x : (useb ? vb.x : vc.x), inner ? vi.y : (useb ? vb.y : vc.y),
                  inner ? vi.z : (useb ? vb.z : vc.z)};
  double m0 = inner ? la : (useb ? b0 : c0), mb = inner ? lb : (useb ? b1 : 0.0), mc = inner ? lc : (useb ? 0.0 : c1);
  unsigned mask = inner ? 7u : (useb ? kb : kc);  // bits 0, 1, 2: a, b, c
  if (pt) v = a, m0 = 1.0, mb = mc = 0.0, mask = 1u;
  // the best of the faces that count, in order
  const double nv = norm2(v);
  const double n0 = quad_get<kQuad0>(nv), n1 = quad_get<kQuad1>(nv), n2 = quad_get<kQuad2>(nv);
  uint32_t f = (faces & 1u) ? 0u : ((faces & 2u) ? 1u : 2u);
  double nb = f == 0 ? n0 : (f == 1 ? n1 : n2);
  if (f < 1 && (faces & 2u) && n1 < nb) f = 1, nb = n1;
  if (f < 2 && (faces & 4u) && n2 < nb) f = 2;
  const int src = (int)((__lane_id() & ~3u) | f);
  best.v = {__shfl(v.x, src), __shfl(v.y, src), __shfl(v.z, src)};
  m0 = __shfl(m0, src);
  mb = __shfl(mb, src);
  mc = __shfl(mc, src);
  mask = (unsigned)__shfl((int)mask, src);
  best.lam[0] = m0;
  best.lam[1] = f == 0 ? 0.0 : mb;
  best.lam[2] = f == 0 ? mb : (f == 2 ? mc : 0.0);
  best.lam[3] = f == 2 ? 0.0 : mc;
  best.mask = (mask & 1u) | ((mask & 2u) ? (f == 0 ? 4u : 2u) : 0u) | ((mask & 4u) ? (f == 2 ? 4u : 8u) : 0u);
  if (in) {
    best.v = {0.0, 0.0, 0.0};
    best.lam[0] = l0;
    best.lam[1] = l1;
    best.lam[2] = l2;
    best.lam[3] = l3;
    best.mask = 15u;
  }
  return best;
}

// MODE 0: the entries the screen queued (FP64 path).  MODE 1: the FP64
// re-runs of the FP32-mixed path, each started from the direction its FP32
// search ended on (left in its result slot; a zero direction starts cold):
// near the optimum already, and meeting the same FP64 gap test.
//
// What bounds it is FP64 issue on a long queue -- a superquadric support is
// seven pow calls of ~210 instructions, ~800 cycles each however many waves
// share the SIMD -- and the chain of a search's iterations on a short one
// (~10 cycles per dependent FP64 instruction, tens of iterations).  A long
// queue therefore takes one lane per entry (L = 1); a short one four: two per
// body, which take the independent pow calls of a support side by side, one
// per face of the simplex (L = 4).  Four lanes issue about twice the
// instructions per entry: the line lies where one lane per entry begins to fill
// the waves.  Touching superquadrics, ms by four and by one: 28,000 entries
// 0.364 and 0.805, 46,000 0.46 and 0.80, 69,000 0.80 and 0.88, 80,000 0.82 and
// 0.81, 98,000 0.99 and 0.82, 127,000 1.23 and 0.85, 173,000 1.60 and 1.08 (the
// two meet at 80,000, below the line).
//
// A lane whose search has ended waits until a quarter of the wave's entries
// have, then those store their results and take the next entries together
// (finishing and setting up cost the wave the same for one lane as for all).
// Entries are dealt out evenly at first -- a short queue gives a wave one or
// two, whose lanes take few branches -- and the rest of a long queue goes
// out through a counter.  The simplex points live in LDS, addressed by slot,
// so dropping points reorders slot numbers instead of moving 40 doubles
// through selects; with them the search fits the registers of two waves per
// SIMD.  Measured against two lanes per entry with the points in registers
// (256 VGPRs + up to 188 AGPRs, one wave per SIMD): touching superquadrics
// 0.80 -> 0.56 ms (46,700 searches of 38 iterations), 1.63 -> 1.10 ms
// (173,000 of 32), 600 ellipsoid contacts 0.27 -> 0.185 ms, 600 hull contacts
// 0.128 -> 0.080 ms (both bound by the longest search).
constexpr uint32_t kSearchQuad = 98304;  // longest queue taken by four lanes per entry
template <int MODE, int L>
__device__ __forceinline__ void search64(const DevScene& d, const uint32_t E, double (*pts)[9][64]) {
  using T = double;
  constexpr uint32_t NE = 64 / L;           // entries a wave holds
  // (doubles per simplex point in LDS: the difference, the lane's body's
  // point; L = 1: both bodies')
  const uint32_t W = gridDim.x, w = blockIdx.x;  // one wave per block
  if (w >= E) return;
  const uint32_t lane = threadIdx.x, slot = lane / L;
  const bool odd = L == 4 && (lane & 2u);  // L = 4: the lane's body is B
  const bool lead = lane % L == 0;
  const uint32_t per = min(NE, (E + W - 1) / W);
  const bool nesterov = (d.flags & GRAINS_NESTEROV) != 0;
  const double rel_arg = MODE == 1 ? d.gjk_rel64 : d.gjk_rel;
  const T rel = rel_arg > 0 ? rel_arg : Eps<T>::LOW;
  PairRes<double>* res64 = (PairRes<double>*)d.pair_res;
  PairRes<float>* res32 = (PairRes<float>*)d.pair_res;
  const bool store64 = MODE == 0 || d.res64;
  const V3<T> zero = {T(0), T(0), T(0)};
  auto get = [&](uint32_t s, int c) { return V3<T>{pts[s][c][lane], pts[s][c + 1][lane], pts[s][c + 2][lane]}; };
  auto put = [&](uint32_t s, int c, V3<T> a) {
    pts[s][c][lane] = a.x;
    pts[s][c + 1][lane] = a.y;
    pts[s][c + 2][lane] = a.z;
  };
  auto swap = [&](V3<T> a) { return quad_get<kQuadXor2>(a); };

  uint32_t c_gjk = 0, c_it = 0, c_deep = 0, c_bk = 0, c_maxit = 0;
  // the lane's search
  uint32_t e = 0;
  bool active = false, done = true;  // active: holds an entry; done: its search has ended
  bool dealt = slot >= per;          // its first, dealt entry is taken
  Tr<T> b2a;
  uint32_t shA = 0, shB = 0;         // the bodies' shapes
  // L = 4: the lane's body held in registers (a load per turn is a round
  // trip in the search's chain)
  int kind = 0, nv = 0;
  const T* verts = nullptr;
  T dims[5] = {T(0), T(0), T(0), T(0), T(0)};
  SqPow pw = {};
  uint32_t order = 0;                // slots of the simplex points, newest first, a byte each
  int ns = 0, num_iter = 0;
  T lam[4] = {T(0), T(0), T(0), T(0)};
  V3<T> v = zero, dir = zero, wprev = zero, lastA = zero, lastB = zero;  // last support points (L = 4: lastA the body's own)
  T dist = 0, mu = 0, sep_s = 0, sc = 1;
  bool accel = false, inside = false, warm1 = false, stalled = false, separated = false, gjk = false;
  bool more = E > W * per;  // the counter still has entries (wave-uniform)

  for (;;) {
    if (!__any(!done) || (more && (uint32_t)__popcll(__ballot(active && done)) >= max(1u, NE / 4) * L)) {
      if (active && done) {
        // ---- the entry's result (closestPointsRigidBodies from the search's end on) ----
        const uint32_t si = d.pair_i[e], sj = d.pair_j[e];
        const PoseRec pi = d.pk[si], pj = d.pk[sj];
        const ShapeNP<T>&A = d.np64[pi.shape], &B = d.np64[pj.shape];
        const SimGrid& g = d.grids[pi.sim];
        const V3<T> xi = {pi.x, pi.y, pi.z};
        Tr<T> a2w, b2w;
        pair_frames<T>(g, xi, Qt<T>{pi.qx, pi.qy, pi.qz, pi.qw}, V3<T>{pj.x, pj.y, pj.z},
                       Qt<T>{pj.qx, pj.qy, pj.qz, pj.qw}, a2w, b2w);
        CInfo<T> ci = no_contact<T>();
        uint32_t flag = kFlagCand;
        if (gjk) {
          flag |= kFlagGjk;
          const T ctSum = A.crust + B.crust;
          const bool deep = inside || dist <= Eps<T>::HIGH;
          const T inv = T(1) / sc;
          V3<T> p = lastA, q = lastB;
          if (ns > 0) {
            p = q = zero;
#pragma unroll
            for (int i = 0; i < 4; ++i)
              if (i < ns) {
                const uint32_t s = (order >> (8 * i)) & 3u;
                p = p + lam[i] * get(s, 3);
                if constexpr (L == 1) q = q + lam[i] * get(s, 6);
              }
          }
          p = inv * p;
          if constexpr (L == 1) {
            q = inv * q;
          } else {
            const V3<T> o = swap(p), m = p;
            p = {odd ? o.x : m.x, odd ? o.y : m.y, odd ? o.z : m.z};
            q = {odd ? m.x : o.x, odd ? m.y : o.y, odd ? m.z : o.z};
          }
          T distance = inv * dist - ctSum;
          if (deep) distance = -ctSum;
          if (!separated && !(distance > T(0))) {
            const V3<T> ptA = apply(a2w, p), ptB = apply(b2w, q);
            ci.cp = (ptA + ptB) / T(2);
            V3<T> cv = ptA - ptB;
            if (deep) {
              flag |= kFlagDeep;
              cv = a2w.o - b2w.o;
              ci.cp = (a2w.o + b2w.o) / T(2);
            }
            cv = cv / norm(cv);
            cv = round_tol(cv, Eps<T>::MID);
            ci.cv = (-distance) * cv;
            ci.overlap = distance;
            if (MODE == 0 && d.gjk_rec && lead)
              d.gjk_rec[e] = {{p.x, p.y, p.z}, {q.x, q.y, q.z}, inv * dist, deep ? 1.0 : 0.0};
          }
        } else if (A.kind == GRAINS_SPHERE && B.kind == GRAINS_SPHERE) {
          ci = cp_spheres(A.rc, B.rc, a2w, b2w);
        }
        if (ci.overlap < T(0)) {
          flag |= kFlagContact | slot_bits(g, xi, V3<T>{pj.x, pj.y, pj.z});
          PairRes<T> r;
          contact_force<T, T>(d, g, si, sj, A.material, B.material, A.mass, B.mass, xi, a2w.o,
                              b2w.o, ci, r);
          if (lead) {
            if (store64) {
              res64[e] = r;
            } else {
              PairRes<float> h;
#pragma unroll
              for (int k = 0; k < 3; ++k) h.f[k] = (float)r.f[k], h.m[k] = (float)r.m[k];
              res32[e] = h;
            }
          }
        }
        if (lead) {
          d.pair_flag[e] = MODE == 1 ? flag | kFlagRefine : flag;
          c_gjk += gjk;
          c_it += num_iter;
          c_maxit = c_maxit > (uint32_t)num_iter ? c_maxit : (uint32_t)num_iter;
          c_deep += (flag & kFlagDeep) != 0;
          c_bk += gjk && stalled;
        }
        active = false;
      }
      // ---- the next entries ----
      uint32_t k = ~0u;
      if (!active && !dealt) {
        dealt = true;
        k = w + W * slot;
      } else if (more) {
        const bool want = !active && slot < per;
        const uint64_t m = __ballot(want && lead);
        if (m) {
          uint32_t base = 0;
          if (lane == 0) base = W * per + atomicAdd(d.queue_next, (uint32_t)__popcll(m));
          base = __shfl(base, 0);
          if (base + (uint32_t)__popcll(m) >= E) more = false;
          if (want) k = base + (uint32_t)__popcll(m & ((1ull << (lane - lane % L)) - 1ull));
        }
      }
      if (k < E) {
        e = MODE == 0 ? defer_entry(d, k) : d.refine_list[k];
        active = true;
        const uint32_t si = d.pair_i[e], sj = d.pair_j[e];
        const PoseRec pi = d.pk[si], pj = d.pk[sj];
        shA = pi.shape;
        shB = pj.shape;
        const ShapeNP<T>&A = d.np64[shA], &B = d.np64[shB];
        Tr<T> a2w, b2w;
        pair_frames<T>(d.grids[pi.sim], V3<T>{pi.x, pi.y, pi.z}, Qt<T>{pi.qx, pi.qy, pi.qz, pi.qw},
                       V3<T>{pj.x, pj.y, pj.z}, Qt<T>{pj.qx, pj.qy, pj.qz, pj.qw}, a2w, b2w);
        if constexpr (L == 4) {
          const ShapeNP<T>& C = odd ? B : A;
          kind = C.kind;
          nv = C.nv;
          verts = d.cverts64 + 3 * (size_t)C.voff;
#pragma unroll
          for (int k5 = 0; k5 < 5; ++k5) dims[k5] = C.core[k5];
          pw = d.sq64[odd ? shB : shA];
        }
        done = true;
        gjk = inside = warm1 = stalled = separated = false;
        num_iter = 0;
        ns = 0;
        const T rsum = A.rc + B.rc;
        if (!(A.kind == GRAINS_SPHERE && B.kind == GRAINS_SPHERE) && norm(b2w.o - a2w.o) - rsum < T(0) &&
            obb_intersect(A.bbox, B.bbox, a2w, b2w)) {
          gjk = true;
          done = false;
          b2a = relative(a2w, b2w);
          int ex;
          frexp(rsum, &ex);
          sc = ldexp(T(1), -ex);
          b2a.o = sc * b2a.o;
          sep_s = sc * (A.crust + B.crust);
          v = -b2a.o;
          dist = norm(v);
          mu = T(0);
          dir = v;
          wprev = v;
          lastA = lastB = zero;
          accel = nesterov;
          if (MODE == 1) {
            V3<T> start;
            if (store64) {
              const PairRes<double> q = res64[e];
              start = {q.f[0], q.f[1], q.f[2]};
            } else {
              const PairRes<float> q = res32[e];
              start = {(T)q.f[0], (T)q.f[1], (T)q.f[2]};
            }
            const T nn = dot(start, start);
            if (nn > T(0) && nn < INFINITY) {
              warm1 = true;
              accel = false;
              dir = vm(start, a2w.R);  // into A's frame
            }
          }
        }
      }
      if (!__any(active)) break;  // every lane has stored its last result
    }
    // ---- one iteration ----
    if (done) continue;
    if (!warm1 && !(dist > Eps<T>::HIGH && num_iter < kGjkMaxIter)) {
      if (dist > Eps<T>::HIGH) stalled = true;  // out of iterations
      done = true;
      continue;
    }
    // the simplex, read ahead of its use after the supports (L = 4: the two
    // older points of the lane's face)
    V3<T> y[4];
    if constexpr (L == 4) {
      y[1] = get((order >> ((lane & 3u) == 0 ? 8 : 0)) & 3u, 0);
      y[2] = get((order >> ((lane & 3u) < 2 ? 16 : 8)) & 3u, 0);
    } else {
#pragma unroll
      for (int i = 0; i < 3; ++i) y[i + 1] = i < ns ? get((order >> (8 * i)) & 3u, 0) : zero;
    }
    V3<T> sd = warm1 ? dir : v;
    if (accel && num_iter >= kNesterovIters) accel = false;
    if (accel) {
      const T delta = T(num_iter + 1) / T(num_iter + 3);
      const V3<T> yk = delta * v + (T(1) - delta) * wprev;
      const T ny = norm(yk), nd = norm(dir);
      if (num_iter != 0 && ny > Eps<T>::HIGH && nd > Eps<T>::HIGH)
        sd = (delta / nd) * dir + ((T(1) - delta) / ny) * yk;
      dir = sd;
    }
    if constexpr (L == 4) {
      const V3<T> rb = vm(sd, b2a.R);
      const V3<T> in = {odd ? rb.x : -sd.x, odd ? rb.y : -sd.y, odd ? rb.z : -sd.z};
      V3<T> r;
      if (kind == GRAINS_SUPERQUADRIC) {
        r = sq_support_split<true>(dims, pw, in);
      } else if (kind == GRAINS_POLYHEDRON) {
        r = poly_support_split(verts, nv, in);
      } else {
        SupCtx<T> c;
        c.kind = kind;
        c.nv = nv;
        c.d = dims;
        c.verts = verts;
        r = support(c, in);
      }
      lastA = sc * r;
    } else {
      // A's support, then B's, through one copy of the code
#pragma unroll 1
      for (int body = 0; body < 2; ++body) {
        const uint32_t sh = body ? shB : shA;
        const ShapeNP<T>& C = d.np64[sh];
        const V3<T> in = body ? vm(sd, b2a.R) : -sd;
        V3<T> r;
        if (C.kind == GRAINS_SUPERQUADRIC) {
          r = sq_support_split<false>(C.core, d.sq64[sh], in);
        } else {
          SupCtx<T> c;
          c.kind = C.kind;
          c.nv = C.nv;
          c.d = C.core;
          c.verts = d.cverts64 + 3 * (size_t)C.voff;
          r = support(c, in);
        }
        r = sc * r;
        if (body)
          lastB = r;
        else
          lastA = r;
      }
    }
    V3<T> wv;
    if constexpr (L == 1) {
      wv = lastA - apply(b2a, lastB);
    } else {
      const V3<T> o = swap(lastA);
      wv = (odd ? o : lastA) - apply(b2a, odd ? lastA : o);
    }
    // the new point's place is worked out beside the tests that may end the
    // search without it: their divisions overlap
    const T lb = dot(sd, wv) / (warm1 || accel ? norm(sd) : dist);
    if (mu < lb) mu = lb;
    y[0] = wv;
    bool degen = false;
    SvBest q;
    if constexpr (L == 4) {
      // lane 0 holds points 2 and 3, lane 1 points 1 and 3
      const uint32_t l4 = lane & 3u;
      const bool dup = (same(y[1], wv) && ns >= (l4 == 0 ? 2 : 1)) || (same(y[2], wv) && ns >= (l4 < 2 ? 3 : 2));
      degen = ((__ballot(dup) >> (lane & ~3u)) & 0xfull) != 0;
      q = sv_closest_quad(wv, y[1], y[2], ns + 1);
    } else {
#pragma unroll
      for (int i = 0; i < 3; ++i)
        if (i < ns && same(y[i + 1], wv)) degen = true;
      q = sv_closest(y, ns + 1);
    }
    const T nd = norm(q.v);
    if (mu > sep_s) {
      separated = true;
      done = true;
    } else if (!warm1 && dist - mu <= dist * rel) {
      done = true;
    } else {
      bool progress = false;
      if (!degen) {
        ++num_iter;
        inside = q.mask == 15u;
        progress = inside || num_iter <= 1 || nd < dist;
      }
      if (progress) {
        // a slot none of the (at most three) points holds
        uint32_t used = 0;
#pragma unroll
        for (int i = 0; i < 3; ++i)
          if (i < ns) used |= 1u << ((order >> (8 * i)) & 3u);
        const uint32_t fresh = (uint32_t)__ffs(~used) - 1u;
        put(fresh, 0, wv);
        put(fresh, 3, lastA);
        if constexpr (L == 1) put(fresh, 6, lastB);
        const uint32_t all = (order << 8) | fresh;
        order = 0;
        ns = 0;
#pragma unroll
        for (int i = 0; i < 4; ++i)
        {
          const bool on = (q.mask >> i) & 1u;
          order |= on ? ((all >> (8 * i)) & 3u) << (8 * ns) : 0u;
#pragma unroll
          for (int k = 0; k <= i; ++k) lam[k] = on && ns == k ? q.lam[i] : lam[k];
          ns += on ? 1 : 0;
        }
        wprev = wv;
        v = q.v;
        dist = inside ? T(0) : nd;
        if (inside || (warm1 && dist - mu <= dist * rel)) done = true;
      } else if (accel) {
        // rounding has the last word (a repeated point, or |v| no smaller):
        // an accelerated search goes on without momentum, a plain one ends
        // with the simplex it has
        accel = false;
      } else {
        stalled = true;
        done = true;
      }
      warm1 = false;
    }
  }
  if (MODE == 0) {
    count_add(d.counters, kCntGjk, c_gjk);
    count_add(d.counters, kCntGjkIters, c_it);
    count_add(d.counters, kCntDeep, c_deep);
    count_add(d.counters, kCntBackup, c_bk);
    count_max(d.counters, kCntMaxIters, c_maxit);
  } else {
    count_add(d.counters, kCntRefIters, c_it);
    count_max(d.counters, kCntRefMaxIters, c_maxit);
  }
}

template <int MODE>
__global__ void __launch_bounds__(64) __attribute__((amdgpu_waves_per_eu(2, 2))) k_search64(DevScene d) {
  __shared__ double pts[4][9][64];
  const uint32_t E = MODE == 0 ? defer_total(d) : *d.refine_count;
  if (E <= kSearchQuad)
    search64<MODE, 4>(d, E, pts);
  else
    search64<MODE, 1>(d, E, pts);
}

}  // namespace gr
