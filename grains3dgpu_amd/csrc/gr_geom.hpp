// gr_geom.hpp -- narrow phase of the DEM step on the device: support maps,
// oriented-bounding-box test, GJK distance (Johnson's sub-algorithm for the
// reference semantics, signed volumes for the physics semantics), contact
// dispatch and the Hooke spring-dashpot / Coulomb force.
//
// Everything is templated on the arithmetic type T (double for the plain
// path, float for the FP32-mixed path).  The Johnson sub-algorithm keeps its
// determinant cache det[16][4] and dot products dp[4][4] in registers: every
// index is made a compile-time constant (the free slot `last` is dispatched
// to one of four instantiations, subsets are enumerated with fold
// expressions), so no private-memory scratch is needed per lane.
#pragma once

#include <utility>

#include "../../include/grains_hip.h"
#include "gr_math.hpp"

#define GR_D __device__ __forceinline__

namespace gr {

// Narrow-phase view of one shape (per particle or obstacle).
template <class T>
struct alignas(16) ShapeNP {
  int32_t kind, material, nv, voff;
  T dims[5];   // full shape
  T core[5];   // crust core (physics semantics)
  T crust;
  T rc;        // circumscribed radius used by the bounding-sphere test
  T bbox[3];   // OBB half extents (BoundingBox of the full shape)
  T mass;
  T rc_max;    // largest distance of the full shape from its origin (>= rc
               // of either semantics): bounds every support point
  T pad;
};

// Hooke parameters with the precomputed m_muen (HookeContactForceModel.cpp:56).
template <class T>
struct HookeP {
  T kn, en, etat, muc, kr, muen;
};

struct GjkArgs {
  uint32_t flags;
  double rel;   // relative tolerance of the optimality gap
};

// ---- support maps -----------------------------------------------------------
// sgn (MiscMath.hh:68-72)
template <class T> GR_D T sgn(T x) { return T((T(0) < x) - (x < T(0))); }

// Superquadric::support (Superquadric.cpp:169-205), the reference's pow chain.
// An ellipsoid (n1 = n2 = 2) takes the chain with its exponents resolved:
// every one is exactly 1, 0, 2 or 1/2, so pow(x, 1) = x, pow(x, 0) = 1,
// pow(x, 2) = x x and pow(x, 1/2) = sqrt(x), the last two rounded once
// (correctly), with the chain's operands in its order -- a few operations
// instead of seven pow calls per support.
template <class T>
GR_D V3<T> sq_support_pow(const T* d, V3<T> v) {
  const T a = d[0], b = d[1], c = d[2], n1 = d[3], n2 = d[4];
  const T ax = fabs(v.x), ay = fabs(v.y), az = fabs(v.z);
  const T sx = sgn(v.x), sy = sgn(v.y), sz = sgn(v.z);
  if (n1 == T(2) && n2 == T(2)) {
    if (ax == T(0)) {
      if (ay == T(0)) return {T(0), T(0), sz * c};
      const T alpha = c / b * az / ay;
      const T yt = T(1) / sqrt(T(1) + alpha * alpha);
      return {T(0), sy * b * yt, sz * alpha * c * yt};
    }
    const T alpha = b / a * ay / ax;
    const T temp = T(1) + alpha * alpha;
    const T beta = c / a * az / ax;  // gamma = pow(temp, 0) = 1
    const T xt = T(1) / sqrt(temp + beta * beta);
    return {sx * a * xt, sy * alpha * b * xt, sz * beta * c * xt};
  }
  if (ax == T(0)) {
    if (ay == T(0)) return {T(0), T(0), sz * c};
    T alpha = pow(c / b * az / ay, T(1) / (n1 - T(1)));
    T yt = T(1) / pow(T(1) + pow(alpha, n1), T(1) / n1);
    return {T(0), sy * b * yt, sz * alpha * c * yt};
  }
  // (independent pow calls side by side: their instruction chains interleave,
  // five in sequence instead of seven)
  const T alpha = pow(b / a * ay / ax, T(1) / (n2 - T(1)));
  const T zeta = pow(c / a * az / ax, T(1) / (n1 - T(1)));
  const T temp = T(1) + pow(alpha, n2);
  const T gamma = pow(temp, (n1 - n2) / (n2 * (n1 - T(1))));
  const T tr = pow(temp, n1 / n2);
  const T beta = gamma * zeta;
  const T xt = T(1) / pow(tr + pow(beta, n1), T(1) / n1);
  return {sx * a * xt, sy * alpha * b * xt, sz * beta * c * xt};
}

// native v_exp_f32 / v_log_f32 (base 2, about 1 ulp)
GR_D float fexp2(float x) { return __builtin_amdgcn_exp2f(x); }
GR_D float flog2(float x) { return __builtin_amdgcn_logf(x); }

// Per-shape constants of the FP32 log-domain superquadric support.
struct SqLog {
  float la, lb, lc;        // log2 of the semi-axes
  float n1, n2, k1, k2, g, r, in1;
};
GR_D SqLog sq_log_prepare(const float* d) {
  SqLog s;
  s.la = flog2(d[0]);
  s.lb = flog2(d[1]);
  s.lc = flog2(d[2]);
  s.n1 = d[3];
  s.n2 = d[4];
  s.k1 = 1.0f / (d[4] - 1.0f);                       // 1/(n2-1)
  s.k2 = 1.0f / (d[3] - 1.0f);                       // 1/(n1-1)
  s.g = (d[3] - d[4]) / (d[4] * (d[3] - 1.0f));     // (n1-n2)/(n2(n1-1))
  s.r = d[3] / d[4];                                 // n1/n2
  s.in1 = 1.0f / d[3];
  return s;
}
// log2(1 + 2^e), overflow-free
GR_D float softplus2(float e) {
  return e > 0.0f ? e + flog2(1.0f + fexp2(-e)) : flog2(1.0f + fexp2(e));
}
// log2(2^a + 2^b)
GR_D float logadd2(float a, float b) {
  float m = fmaxf(a, b);
  return m + flog2(1.0f + fexp2(-fabsf(a - b)));
}
// Same closed form as sq_support_pow, evaluated in the log2 domain with the
// native v_log_f32 / v_exp_f32: 10 transcendentals instead of 7 pow, and no
// overflow of alpha^n2 for near-axis directions.
GR_D V3<float> sq_support_log(const SqLog& s, V3<float> v) {
  const float ax = fabsf(v.x), ay = fabsf(v.y), az = fabsf(v.z);
  const float sx = sgn(v.x), sy = sgn(v.y), sz = sgn(v.z);
  if (ax == 0.0f) {
    if (ay == 0.0f) return {0.0f, 0.0f, sz * fexp2(s.lc)};
    float La = (s.lc - s.lb + flog2(az) - flog2(ay)) * s.k2;
    float Lyt = -s.in1 * softplus2(s.n1 * La);
    return {0.0f, sy * fexp2(s.lb + Lyt), sz * fexp2(s.lc + La + Lyt)};
  }
  const float lx = flog2(ax);
  float La = (s.lb - s.la + flog2(ay) - lx) * s.k1;
  float Lt = softplus2(s.n2 * La);
  float Lb = Lt * s.g + (s.lc - s.la + flog2(az) - lx) * s.k2;
  float Lxt = -s.in1 * logadd2(Lt * s.r, s.n1 * Lb);
  return {sx * fexp2(s.la + Lxt), sy * fexp2(s.lb + La + Lxt), sz * fexp2(s.lc + Lb + Lxt)};
}

// Per-lane shape context for GJK: which dims, and FP32 log constants.
template <class T>
struct SupCtx {
  int kind, nv;
  const T* d;           // dims in use (full or core)
  const T* verts;       // polyhedron vertices in use (x,y,z triplets)
  SqLog lg;             // used when T = float and kind = SUPERQUADRIC
};

template <class T>
GR_D SupCtx<T> sup_ctx(const ShapeNP<T>& s, bool core, const T* verts_full, const T* verts_core) {
  SupCtx<T> c;
  c.kind = s.kind;
  c.nv = s.nv;
  c.d = core ? s.core : s.dims;
  c.verts = (core ? verts_core : verts_full) + 3 * (size_t)s.voff;
  if constexpr (sizeof(T) == 4) {
    if (s.kind == GRAINS_SUPERQUADRIC) c.lg = sq_log_prepare(c.d);
  }
  return c;
}

// A's context on even lanes, B's on odd ones, field by field
template <class T>
GR_D SupCtx<T> lane_ctx(bool odd, const SupCtx<T>& A, const SupCtx<T>& B) {
  SupCtx<T> c;
  c.kind = odd ? B.kind : A.kind;
  c.nv = odd ? B.nv : A.nv;
  c.d = odd ? B.d : A.d;
  c.verts = odd ? B.verts : A.verts;
  if constexpr (sizeof(T) == 4) c.lg = odd ? B.lg : A.lg;
  return c;
}

// Sphere.cpp:111-114, Box.cpp:129-134, Rectangle.cpp:115-120,
// Superquadric.cpp:169-205, Cylinder.cpp:118-131 (dims r, h/2),
// Cone.cpp:126-141 (dims r, h/4, sine of the half angle); polyhedron: first
// vertex maximising v.x.
// The cylinder's and cone's test for a direction along the axis compares
// |(v_x, v_z)| with EPS in the caller's length units; GJK directions are
// differences of points, ~1e-6..1e-3 in SI for millimetre grains, so FP32
// takes the FP64 value 1e-10 (FP32's 1e-5 would send most directions to the
// axis point).
template <class T>
GR_D V3<T> support(const SupCtx<T>& c, V3<T> v) {
  const T* d = c.d;
  constexpr T kAxisEps = T(Eps<double>::MID);
  switch (c.kind) {
    case GRAINS_SPHERE: {
      T n = norm(v);
      return d[0] * (v / n);
    }
    case GRAINS_BOX:
      return {v.x < T(0) ? -d[0] : d[0], v.y < T(0) ? -d[1] : d[1], v.z < T(0) ? -d[2] : d[2]};
    case GRAINS_SUPERQUADRIC:
      if constexpr (sizeof(T) == 4)
        return sq_support_log(c.lg, v);
      else
        return sq_support_pow(d, v);
    case GRAINS_RECTANGLE:
      return {v.x < T(0) ? -d[0] : d[0], v.y < T(0) ? -d[1] : d[1], T(0)};
    case GRAINS_CYLINDER: {
      const T s = sqrt(v.x * v.x + v.z * v.z);
      const T hy = v.y < T(0) ? -d[1] : d[1];
      if (s > kAxisEps) {
        const T k = d[0] / s;
        return {v.x * k, hy, v.z * k};
      }
      return {T(0), hy, T(0)};
    }
    case GRAINS_CONE: {
      if (v.y > norm(v) * d[2]) return {T(0), T(3) * d[1], T(0)};
      const T s = sqrt(v.x * v.x + v.z * v.z);
      if (s > kAxisEps) {
        const T k = d[0] / s;
        return {v.x * k, -d[1], v.z * k};
      }
      return {T(0), -d[1], T(0)};
    }
    case GRAINS_POLYHEDRON: {
      const T* P = c.verts;
      V3<T> best = {P[0], P[1], P[2]};
      T bd = dot(v, best);
      for (int i = 1; i < c.nv; ++i) {
        V3<T> p = {P[3 * i], P[3 * i + 1], P[3 * i + 2]};
        T dd = dot(v, p);
        if (dd > bd) {
          bd = dd;
          best = p;
        }
      }
      return best;
    }
  }
  return {T(0), T(0), T(0)};
}

// ---- OBB, Grains/CollisionDetection/src/OBB.cpp:32-94 -----------------------
template <class T>
GR_D bool obb_intersect(const T* a, const T* b, const Tr<T>& A, const Tr<T>& B) {
  const T LO = Eps<T>::LOW;
  M3<T> ori = transpose(A.R);
  V3<T> c3 = mv(ori, B.o - A.o);
  ori = mmul(ori, B.R);
  const T cen[3] = {c3.x, c3.y, c3.z};
  T o[3][3], oa[3][3];
#pragma unroll
  for (int i = 0; i < 3; ++i)
#pragma unroll
    for (int j = 0; j < 3; ++j) {
      o[i][j] = ori.m[3 * i + j];
      oa[i][j] = fabs(o[i][j]) + LO;
    }
  bool sep = false;
#pragma unroll
  for (int i = 0; i < 3; ++i)
    sep |= fabs(cen[i]) > (a[i] + b[0] * oa[i][0] + b[1] * oa[i][1] + b[2] * oa[i][2]);
#pragma unroll
  for (int i = 0; i < 3; ++i)
    sep |= fabs(cen[0] * o[0][i] + cen[1] * o[1][i] + cen[2] * o[2][i]) >
           (b[i] + a[0] * oa[0][i] + a[1] * oa[1][i] + a[2] * oa[2][i]);
#pragma unroll
  for (int j = 0; j < 3; ++j)
#pragma unroll
    for (int i = 0; i < 3; ++i) {
      const int i1 = (i + 1) % 3, i2 = (i + 2) % 3, j1 = (j + 1) % 3, j2 = (j + 2) % 3;
      sep |= fabs(cen[i2] * o[i1][j] - cen[i1] * o[i2][j]) >
             (a[i1] * oa[i2][j] + a[i2] * oa[i1][j] + b[j1] * oa[i][j2] + b[j2] * oa[i][j1]);
    }
  return !sep;
}

// ---- Johnson's distance sub-algorithm (GJK_JH.cpp:9-207) ----------------------
template <class T>
struct JH {
  V3<T> y[4], p[4], q[4];
  T det[16][4];
  T dp[4][4];
};

template <class T, int S>
GR_D bool jh_valid(const JH<T>& st, unsigned all_bits) {
  bool ok = true;
#pragma unroll
  for (int i = 0; i < 4; ++i) {
    const unsigned bit = 1u << i;
    if (all_bits & bit) {
      if (S & bit) {
        if (st.det[S][i] <= Eps<T>::MID) ok = false;
      } else if (st.det[S | bit][i] > T(0)) {
        ok = false;
      }
    }
  }
  return ok;
}

template <class T, int S>
GR_D bool jh_proper(const JH<T>& st) {
  bool ok = true;
#pragma unroll
  for (int i = 0; i < 4; ++i)
    if ((S & (1 << i)) && st.det[S][i] <= Eps<T>::MID) ok = false;
  return ok;
}

template <class T, int S>
GR_D V3<T> jh_vector(const JH<T>& st) {
  T sum = T(0);
  V3<T> v = {T(0), T(0), T(0)};
#pragma unroll
  for (int i = 0; i < 4; ++i)
    if (S & (1 << i)) {
      sum += st.det[S][i];
      v = v + st.det[S][i] * st.y[i];
    }
  return (T(1) / sum) * v;
}

template <class T, int S>
GR_D void jh_points(const JH<T>& st, V3<T>& p1, V3<T>& p2) {
  T sum = T(0);
  p1 = {T(0), T(0), T(0)};
  p2 = {T(0), T(0), T(0)};
#pragma unroll
  for (int i = 0; i < 4; ++i)
    if (S & (1 << i)) {
      sum += st.det[S][i];
      p1 = p1 + st.det[S][i] * st.p[i];
      p2 = p2 + st.det[S][i] * st.q[i];
    }
  T s = T(1) / sum;
  p1 = s * p1;
  p2 = s * p2;
}

template <class T, int... Is>
GR_D void jh_points_dispatch(const JH<T>& st, unsigned bits, V3<T>& p1, V3<T>& p2,
                             std::integer_sequence<int, Is...>) {
  ((bits == unsigned(Is + 1) ? jh_points<T, Is + 1>(st, p1, p2) : void()), ...);
}

// one subset S of `bits` tried in the descending scan of closest()
template <class T, int L, int S>
GR_D void jh_try(const JH<T>& st, unsigned bits, unsigned all_bits, bool& found, unsigned& nb, V3<T>& v) {
  if constexpr ((S & (1 << L)) == 0) {
    if (!found && (unsigned(S) & bits) == unsigned(S)) {
      if (jh_valid<T, S | (1 << L)>(st, all_bits)) {
        nb = S | (1 << L);
        v = jh_vector<T, S | (1 << L)>(st);
        found = true;
      }
    }
  }
}
template <class T, int L, int... Is>
GR_D void jh_try_all(const JH<T>& st, unsigned bits, unsigned all_bits, bool& found, unsigned& nb,
                     V3<T>& v, std::integer_sequence<int, Is...>) {
  (jh_try<T, L, 15 - Is>(st, bits, all_bits, found, nb, v), ...);
}
// backup procedure: best proper subset of all_bits (descending scan)
template <class T, int S>
GR_D void jh_backup1(const JH<T>& st, unsigned all_bits, T& best, unsigned& nb, V3<T>& v) {
  if ((unsigned(S) & all_bits) == unsigned(S)) {
    if (jh_proper<T, S>(st)) {
      V3<T> u = jh_vector<T, S>(st);
      T d2 = norm2(u);
      if (d2 < best) {
        best = d2;
        nb = S;
        v = u;
      }
    }
  }
}
template <class T, int... Is>
GR_D void jh_backup_all(const JH<T>& st, unsigned all_bits, T& best, unsigned& nb, V3<T>& v,
                        std::integer_sequence<int, Is...>) {
  (jh_backup1<T, 15 - Is>(st, all_bits, best, nb, v), ...);
}

// computeDet + closest for the new point in slot L (GJK_JH.cpp:9-63, 143-194)
template <class T, int L>
GR_D bool jh_closest(JH<T>& S, unsigned& bits, unsigned all_bits, V3<T>& v) {
  constexpr unsigned LB = 1u << L;
#pragma unroll
  for (int i = 0; i < 4; ++i)
    if (i != L && (bits & (1u << i))) {
      T d = dot(S.y[i], S.y[L]);
      S.dp[i][L] = d;
      S.dp[L][i] = d;
    }
  S.dp[L][L] = dot(S.y[L], S.y[L]);
  S.det[LB][L] = T(1);
#pragma unroll
  for (int j = 0; j < 4; ++j) {
    if (j == L) continue;
    const unsigned sj = 1u << j;
    if (bits & sj) {
      const unsigned s2 = sj | LB;
      S.det[s2][j] = S.dp[L][L] - S.dp[L][j];
      S.det[s2][L] = S.dp[j][j] - S.dp[j][L];
#pragma unroll
      for (int k = 0; k < j; ++k) {
        if (k == L) continue;
        const unsigned sk = 1u << k;
        if (bits & sk) {
          const unsigned s3 = sk | s2;
          S.det[s3][k] = S.det[s2][j] * (S.dp[j][j] - S.dp[j][k]) + S.det[s2][L] * (S.dp[L][j] - S.dp[L][k]);
          S.det[s3][j] = S.det[sk | LB][k] * (S.dp[k][k] - S.dp[k][j]) +
                         S.det[sk | LB][L] * (S.dp[L][k] - S.dp[L][j]);
          S.det[s3][L] = S.det[sk | sj][k] * (S.dp[k][k] - S.dp[k][L]) +
                         S.det[sk | sj][j] * (S.dp[j][k] - S.dp[j][L]);
        }
      }
    }
  }
  if (all_bits == 15) {
    auto& det = S.det;
    auto& dp = S.dp;
    det[15][0] = det[14][1] * (dp[1][1] - dp[1][0]) + det[14][2] * (dp[2][1] - dp[2][0]) +
                 det[14][3] * (dp[3][1] - dp[3][0]);
    det[15][1] = det[13][0] * (dp[0][0] - dp[0][1]) + det[13][2] * (dp[2][0] - dp[2][1]) +
                 det[13][3] * (dp[3][0] - dp[3][1]);
    det[15][2] = det[11][0] * (dp[0][0] - dp[0][2]) + det[11][1] * (dp[1][0] - dp[1][2]) +
                 det[11][3] * (dp[3][0] - dp[3][2]);
    det[15][3] = det[7][0] * (dp[0][0] - dp[0][3]) + det[7][1] * (dp[1][0] - dp[1][3]) +
                 det[7][2] * (dp[2][0] - dp[2][3]);
  }
  bool found = false;
  unsigned nb = bits;
  jh_try_all<T, L>(S, bits, all_bits, found, nb, v, std::make_integer_sequence<int, 15>{});
  if (found) {
    bits = nb;
    return true;
  }
  if (jh_valid<T, LB>(S, all_bits)) {
    bits = LB;
    v = S.y[L];
    return true;
  }
  T best = T(INFINITY);
  jh_backup_all<T>(S, all_bits, best, nb, v, std::make_integer_sequence<int, 15>{});
  bits = nb;
  return false;
}

// Result of one GJK distance query.
template <class T>
struct GjkOut {
  T dist;
  V3<T> pa, pb;   // witness points in the local frames of A and B
  int iters;
  bool deep;      // physics semantics: crust cores overlap
  bool backup;    // Johnson: the backup procedure was taken; signed volumes:
                  // the search ended on rounding or the cap, not the gap test
  bool separated; // signed volumes: the lower bound passed `sep` (no contact)
  V3<T> vdir;     // signed volumes: the search's last direction in A's frame
                  // (the closest-point direction of a converged search)
  bool has_v;     // vdir is a direction (not inside, not degenerate)
};

// GJK iteration budget of a complete search
constexpr int kGjkMaxIter = 1000;

// computeClosestPoints_GJK_JH (GJK_JH.cpp:310-391), exactly the reference
// (the REF_QUIRKS semantics): full shapes, v0 = s_A(0) - b2a(s_B(0)), the
// break on mu < 1e-4*rel, the stale |v| kept when Johnson's backup procedure
// is taken.  The physics semantics use gjk_sv.
// PAIR: two lanes per pair, as gjk_sv<PAIR>.
template <class T, bool PAIR = false>
GR_D GjkOut<T> gjk_jh(const SupCtx<T>& A, const SupCtx<T>& B, const Tr<T>& a2w, const Tr<T>& b2w,
                      const GjkArgs& args) {
  const T rel = args.rel > 0 ? T(args.rel) : Eps<T>::LOW;
  const T abs_err = T(1.e-4) * rel;
  JH<T> S;
#pragma unroll
  for (int i = 0; i < 16; ++i)
#pragma unroll
    for (int k = 0; k < 4; ++k) S.det[i][k] = T(0);
#pragma unroll
  for (int i = 0; i < 4; ++i)
#pragma unroll
    for (int k = 0; k < 4; ++k) S.dp[i][k] = T(0);
#pragma unroll
  for (int i = 0; i < 4; ++i) S.y[i] = S.p[i] = S.q[i] = {T(0), T(0), T(0)};
  unsigned bits = 0, all_bits = 0;
  int last = 0;
  T mu = T(0);
  int num_iter = 0;
  const Tr<T> b2a = relative(a2w, b2w);
  const V3<T> zero = {T(0), T(0), T(0)};
  // the support pair in directions da (A's frame) and db (B's)
  V3<T> pl, ql;
  auto supports = [&](const V3<T>& da, const V3<T>& db) {
    if constexpr (PAIR) {
      const bool odd = (__lane_id() & 1u) != 0;
      const SupCtx<T> C = lane_ctx(odd, A, B);
      const V3<T> r = support(C, V3<T>{odd ? db.x : da.x, odd ? db.y : da.y, odd ? db.z : da.z});
      const V3<T> o = {__shfl_xor(r.x, 1), __shfl_xor(r.y, 1), __shfl_xor(r.z, 1)};
      pl = {odd ? o.x : r.x, odd ? o.y : r.y, odd ? o.z : r.z};
      ql = {odd ? r.x : o.x, odd ? r.y : o.y, odd ? r.z : o.z};
    } else {
      pl = support(A, da);
      ql = support(B, db);
    }
  };
  supports(zero, zero);
  V3<T> v = pl - apply(b2a, ql);
  T dist = norm(v);
  bool backup = false;
  while (bits < 15 && dist > Eps<T>::HIGH && num_iter < 1000) {
    last = 0;
    unsigned last_bit = 1;
    while (bits & last_bit) {
      ++last;
      last_bit <<= 1;
    }
    supports(-v, vm(v, b2a.R));
    const V3<T> w = pl - apply(b2a, ql);
    const T lb = dot(v, w) / dist;
    if (mu < lb) mu = lb;
    if (dist - mu <= dist * rel || mu < abs_err) break;
    bool degen = false;
#pragma unroll
    for (int i = 0; i < 4; ++i)
      if ((all_bits & (1u << i)) && same(S.y[i], w)) degen = true;
    if (degen) break;
#pragma unroll
    for (int i = 0; i < 4; ++i)
      if (i == last) {
        S.y[i] = w;
        S.p[i] = pl;
        S.q[i] = ql;
      }
    all_bits = bits | last_bit;
    ++num_iter;
    bool ok;
    switch (last) {
      case 0: ok = jh_closest<T, 0>(S, bits, all_bits, v); break;
      case 1: ok = jh_closest<T, 1>(S, bits, all_bits, v); break;
      case 2: ok = jh_closest<T, 2>(S, bits, all_bits, v); break;
      default: ok = jh_closest<T, 3>(S, bits, all_bits, v); break;
    }
    if (!ok) {
      backup = true;
      break;
    }
    dist = norm(v);
  }
  GjkOut<T> out;
  jh_points_dispatch<T>(S, bits, out.pa, out.pb, std::make_integer_sequence<int, 15>{});
  if (bits == 0) {  // reference: computePoints with an empty simplex gives 0 * (1/0)
    const T s = T(1) / T(0);
    out.pa = s * zero;
    out.pb = s * zero;
  }
  out.dist = dist;
  out.iters = num_iter;
  out.deep = false;
  out.backup = backup;
  out.separated = false;
  return out;
}

// ---- signed-volume distance sub-algorithm (physics semantics) -------------------
// The closest point of a simplex of up to four points to the origin, from the
// signs of the origin's barycentric coordinates (ratios of signed volumes and
// areas), after Montanari, Petrinic and Barbieri (ACM TOG 2017).  No absolute
// thresholds: a degenerate feature (zero area or volume) hands over to its
// sub-features, so FP32 and mm-sized grains in SI units need no special care.
// The simplex is kept newest first (y[0] = last support point) and only
// features containing y[0] are candidates.  Every ratio is taken relative to
// the vertex a = y[0]: edges e = y - a are exact for nearby points and the
// coordinates come from products of a with edges (n.(e2 x a), a.(ac x ad)),
// never from cross products of two far-away vertices such as b x c, whose
// cancellation costs eps |a|^2 / |n| once the simplex has shrunk to the
// contact (|e| ~ 1e-6 |a| near convergence); the first coordinate is 1 minus
// the others and the closest point is a + sum lambda_k e_k.  Every index is a
// template constant; compaction is a fixed network of selects, so the
// simplex (y, p, q, lambda: 40 values) lives in registers.
template <class T>
struct SvSimplex {
  V3<T> y[4], p[4], q[4];
  T lam[4];
};
template <class T>
struct SvRes {
  V3<T> v;
  T lam[4];
  unsigned mask;
};
template <class T> GR_D SvRes<T> sv_point(V3<T> v) {
  SvRes<T> r;
  r.v = v;
  r.lam[0] = r.lam[1] = r.lam[2] = r.lam[3] = T(0);
  r.mask = 0;
  return r;
}
template <class T> GR_D SvRes<T> sv_better(const SvRes<T>& a, const SvRes<T>& b) {
  return norm2(b.v) < norm2(a.v) ? b : a;
}

template <class T, int IA, int IB>
GR_D SvRes<T> sv_seg(const SvSimplex<T>& S) {
  const V3<T> a = S.y[IA], b = S.y[IB];
  const V3<T> t = b - a;
  const T tt = dot(t, t);
  if (tt > T(0)) {
    const T l = -dot(a, t) / tt;
    if (l > T(0) && l < T(1)) {
      SvRes<T> r = sv_point<T>(a + l * t);
      r.lam[IA] = T(1) - l;
      r.lam[IB] = l;
      r.mask = (1u << IA) | (1u << IB);
      return r;
    }
    if (l >= T(1)) {
      SvRes<T> r = sv_point<T>(b);
      r.lam[IB] = T(1);
      r.mask = 1u << IB;
      return r;
    }
  }
  SvRes<T> r = sv_point<T>(a);
  r.lam[IA] = T(1);
  r.mask = 1u << IA;
  return r;
}

template <class T, int IA, int IB, int IC>
GR_D SvRes<T> sv_tri(const SvSimplex<T>& S) {
  const V3<T> a = S.y[IA];
  const V3<T> e1 = S.y[IB] - a, e2 = S.y[IC] - a;
  const V3<T> n = cross(e1, e2);
  const T nn = dot(n, n);
  T la = T(0), lb = T(0), lc = T(0);
  if (nn > T(0)) {
    lb = dot(n, cross(e2, a)) / nn;
    lc = dot(n, cross(a, e1)) / nn;
    la = (T(1) - lb) - lc;
    if (la > T(0) && lb > T(0) && lc > T(0)) {
      SvRes<T> r = sv_point<T>((a + lb * e1) + lc * e2);
      r.lam[IA] = la;
      r.lam[IB] = lb;
      r.lam[IC] = lc;
      r.mask = (1u << IA) | (1u << IB) | (1u << IC);
      return r;
    }
  }
  bool ab = !(nn > T(0)) || lc <= T(0), ac = !(nn > T(0)) || lb <= T(0);
  if (!ab && !ac) ab = ac = true;  // only la <= 0 (rounding): keep a's edges
  SvRes<T> best;
  if (ab) best = sv_seg<T, IA, IB>(S);
  if (ac) {
    const SvRes<T> r = sv_seg<T, IA, IC>(S);
    best = ab ? sv_better(best, r) : r;
  }
  return best;
}

template <class T>
GR_D SvRes<T> sv_tet(const SvSimplex<T>& S) {
  const V3<T> a = S.y[0];
  const V3<T> ab = S.y[1] - a, ac = S.y[2] - a, ad = S.y[3] - a;
  const T D = dot(ab, cross(ac, ad));
  T l1 = T(0), l2 = T(0), l3 = T(0);
  if (D != T(0)) {
    l1 = -dot(a, cross(ac, ad)) / D;
    l2 = dot(ab, cross(ad, a)) / D;
    l3 = dot(ab, cross(a, ac)) / D;
    const T l0 = ((T(1) - l1) - l2) - l3;
    if (l0 > T(0) && l1 > T(0) && l2 > T(0) && l3 > T(0)) {
      SvRes<T> r = sv_point<T>({T(0), T(0), T(0)});
      r.lam[0] = l0;
      r.lam[1] = l1;
      r.lam[2] = l2;
      r.lam[3] = l3;
      r.mask = 15u;
      return r;
    }
  }
  bool fb = D == T(0) || l1 <= T(0), fc = D == T(0) || l2 <= T(0), fd = D == T(0) || l3 <= T(0);
  if (!fb && !fc && !fd) fb = fc = fd = true;
  SvRes<T> best;
  if (fb) best = sv_tri<T, 0, 2, 3>(S);
  if (fc) {
    const SvRes<T> r = sv_tri<T, 0, 1, 3>(S);
    best = fb ? sv_better(best, r) : r;
  }
  if (fd) {
    const SvRes<T> r = sv_tri<T, 0, 1, 2>(S);
    best = (fb || fc) ? sv_better(best, r) : r;
  }
  return best;
}

// keep the points of r.mask, newest first, with their weights: output slot k
// takes the (k+1)-th kept input slot i >= k
template <class T>
GR_D void sv_compact(SvSimplex<T>& S, int& n, const SvRes<T>& r) {
  SvSimplex<T> N = S;
  int c = 0;
#pragma unroll
  for (int i = 0; i < 4; ++i) {
    const bool on = (r.mask >> i) & 1u;
#pragma unroll
    for (int k = 0; k <= i; ++k)
      if (on && c == k) {
        N.y[k] = S.y[i];
        N.p[k] = S.p[i];
        N.q[k] = S.q[i];
        N.lam[k] = r.lam[i];
      }
    c += on ? 1 : 0;
  }
  S = N;
  n = c;
}

// Momentum is applied to this many support points, then plain GJK: on
// superquadric pairs this takes about 20 % fewer iterations than plain GJK,
// with a worst case no worse; uncapped, the momentum zig-zags near the
// optimum and can reach the iteration cap.
constexpr int kNesterovIters = 8;

// GJK with the signed-volume sub-algorithm, physics semantics: crust cores
// (chosen by the caller's support contexts), the pair's unit frame (power of
// two sc with rsum * sc in [0.5, 1)), v0 = centre difference, the
// van den Bergen gap test, NESTEROV momentum on the first kNesterovIters
// support directions (Montaut et al. 2022).  `backup` reports a search that
// ended on rounding (a repeated support point or no decrease of |v|) or on
// the iteration cap instead of the gap test.
// Separation early-out: once the lower bound mu exceeds `sep` (the crust
// sum) the cores are farther apart than the crusts can bridge and the search
// stops with `separated` (INFINITY for a plain distance query).  Contact
// decisions equal those of the full search, which reports no contact exactly
// when its distance, an upper bound, is above sep -- implied by mu > sep.
// warm (optional): a first search direction in A's frame, e.g. the pair's
// closest-point direction of the previous step.  Its support pair seeds the
// simplex (v = w, |v| and the lower bound from it); a search whose gap test
// already holds there ends after that one support pair.  The direction only
// steers the search: the distance, witnesses and decisions meet the same
// gap test as from the centre difference.
// PAIR: two neighbouring lanes (2k, 2k + 1) run the same search on the same
// pair, and each support pair is evaluated half on each: the even lane takes
// A's support, the odd lane B's, and they swap results.  Every step of the
// search is then the same on both lanes, and a search's chain of dependent
// support evaluations is half as long (the FP64 supports of superquadrics
// are chains of pow).
template <class T, bool PAIR = false>
GR_D GjkOut<T> gjk_sv(const SupCtx<T>& A, const SupCtx<T>& B, const Tr<T>& a2w, const Tr<T>& b2w,
                      const GjkArgs& args, T rsum, T sep, const V3<T>* warm = nullptr) {
  const bool nesterov = (args.flags & GRAINS_NESTEROV) != 0;
  const T rel = args.rel > 0 ? T(args.rel) : Eps<T>::LOW;
  Tr<T> b2a = relative(a2w, b2w);
  int ex;
  frexp(rsum, &ex);
  const T sc = ldexp(T(1), -ex);
  b2a.o = sc * b2a.o;
  const T sep_s = sc * sep;
  const V3<T> zero = {T(0), T(0), T(0)};
  SvSimplex<T> S;
#pragma unroll
  for (int i = 0; i < 4; ++i) {
    S.y[i] = S.p[i] = S.q[i] = zero;
    S.lam[i] = T(0);
  }
  int n = 0;
  V3<T> v = -b2a.o, w = zero, pl = zero, ql = zero;
  T dist = norm(v), mu = T(0);
  V3<T> dir = v, wprev = v, last_d = v;
  bool accel = nesterov, inside = false, ran = false, stalled = false, separated = false, done = false;
  int num_iter = 0;
  // the support pair in direction d: pl = s_A(-d), ql = s_B(R^T d) (A's frame, scaled)
  auto supports = [&](const V3<T>& d) {
    if constexpr (PAIR) {
      const bool odd = (__lane_id() & 1u) != 0;
      SupCtx<T> C;  // this lane's shape, field by field
      C.kind = odd ? B.kind : A.kind;
      C.nv = odd ? B.nv : A.nv;
      C.d = odd ? B.d : A.d;
      C.verts = odd ? B.verts : A.verts;
      if constexpr (sizeof(T) == 4) C.lg = odd ? B.lg : A.lg;
      const V3<T> in = odd ? vm(d, b2a.R) : -d;
      const V3<T> r = support(C, in);
      const V3<T> o = {__shfl_xor(r.x, 1), __shfl_xor(r.y, 1), __shfl_xor(r.z, 1)};
      pl = sc * (odd ? o : r);
      ql = sc * (odd ? r : o);
    } else {
      pl = sc * support(A, -d);
      ql = sc * support(B, vm(d, b2a.R));
    }
  };
  if (warm) {
    const V3<T> d0 = *warm;
    last_d = d0;
    supports(d0);
    w = pl - apply(b2a, ql);
    ran = true;
    accel = false;
    const T lb = dot(d0, w) / norm(d0);
    if (mu < lb) mu = lb;
    if (mu > sep_s) {
      separated = true;
      done = true;
    } else {
      S.y[0] = w;
      S.p[0] = pl;
      S.q[0] = ql;
      S.lam[0] = T(1);
      n = 1;
      num_iter = 1;
      v = w;
      dist = norm(w);
      wprev = w;
      dir = w;
      if (dist - mu <= dist * rel) done = true;
    }
  }
  while (!done && dist > Eps<T>::HIGH && num_iter < kGjkMaxIter) {
    V3<T> d = v;
    if (accel && num_iter >= kNesterovIters) accel = false;
    if (accel) {
      const T delta = T(num_iter + 1) / T(num_iter + 3);
      const V3<T> yk = delta * v + (T(1) - delta) * wprev;
      const T ny = norm(yk), nd = norm(dir);
      if (num_iter != 0 && ny > Eps<T>::HIGH && nd > Eps<T>::HIGH)
        d = (delta / nd) * dir + ((T(1) - delta) / ny) * yk;
      dir = d;
    }
    supports(d);
    w = pl - apply(b2a, ql);
    ran = true;
    last_d = d;
    const T lb = accel ? dot(d, w) / norm(d) : dot(v, w) / dist;
    if (mu < lb) mu = lb;
    if (mu > sep_s) {
      separated = true;
      done = true;
      break;
    }
    if (dist - mu <= dist * rel) {
      done = true;
      break;
    }
    bool degen = false;
#pragma unroll
    for (int i = 0; i < 4; ++i)
      if (i < n && same(S.y[i], w)) degen = true;
    if (degen) {
      if (accel) {
        accel = false;
        continue;
      }
      stalled = true;
      done = true;
      break;
    }
    // the simplex holds at most 3 points here (a tetrahedron either encloses
    // the origin or is reduced), so the shift loses nothing and can be undone
#pragma unroll
    for (int i = 3; i > 0; --i) {
      S.y[i] = S.y[i - 1];
      S.p[i] = S.p[i - 1];
      S.q[i] = S.q[i - 1];
      S.lam[i] = S.lam[i - 1];
    }
    S.y[0] = w;
    S.p[0] = pl;
    S.q[0] = ql;
    S.lam[0] = T(0);
    const int n_prev = n;
    n = n + 1;
    ++num_iter;
    SvRes<T> r;
    if (n == 1) {
      r = sv_point<T>(w);
      r.lam[0] = T(1);
      r.mask = 1u;
    } else if (n == 2) {
      r = sv_seg<T, 0, 1>(S);
    } else if (n == 3) {
      r = sv_tri<T, 0, 1, 2>(S);
    } else {
      r = sv_tet<T>(S);
    }
    if (r.mask == 15u) {
      sv_compact(S, n, r);
      inside = true;
      done = true;
      dist = T(0);
      break;
    }
    const T nd = norm(r.v);
    // No progress: rounding has the last word.  Drop w and restore the
    // previous simplex, whose |v| is the best bound found; an accelerated
    // search continues unaccelerated, a plain one stops.  The first support
    // point is exempt: v0 (the centre difference) is not a simplex point.
    if (num_iter > 1 && !(nd < dist)) {
#pragma unroll
      for (int i = 0; i < 3; ++i) {
        S.y[i] = S.y[i + 1];
        S.p[i] = S.p[i + 1];
        S.q[i] = S.q[i + 1];
        S.lam[i] = S.lam[i + 1];
      }
      n = n_prev;
      if (accel) {
        accel = false;
        continue;
      }
      stalled = true;
      done = true;
      break;
    }
    sv_compact(S, n, r);
    wprev = w;
    v = r.v;
    dist = nd;
  }
  // the loop ran out of support points (iteration cap)
  if (!done && dist > Eps<T>::HIGH) stalled = true;
  GjkOut<T> out;
  if (n == 0) {
    out.pa = ran ? pl : zero;
    out.pb = ran ? ql : zero;
  } else {
    V3<T> p = zero, q = zero;
#pragma unroll
    for (int i = 0; i < 4; ++i)
      if (i < n) {
        p = p + S.lam[i] * S.p[i];
        q = q + S.lam[i] * S.q[i];
      }
    out.pa = p;
    out.pb = q;
  }
  const T inv = T(1) / sc;
  out.pa = inv * out.pa;
  out.pb = inv * out.pb;
  out.dist = inv * dist;
  out.iters = num_iter;
  out.deep = inside || dist <= Eps<T>::HIGH;
  out.backup = stalled;
  out.separated = separated;
  // the direction to start from next time: the converged closest-point
  // direction, else the last one searched
  out.vdir = (done && !separated && !inside && n > 0 && dist > Eps<T>::HIGH) ? v : last_d;
  out.has_v = !inside && norm(out.vdir) > T(0);
  return out;
}

// ---- contact information -------------------------------------------------------
template <class T>
struct CInfo {
  V3<T> cp, cv;
  T overlap;
};
template <class T> GR_D CInfo<T> no_contact() { return {{T(0), T(0), T(0)}, {T(0), T(0), T(0)}, T(0)}; }

// closestPointsSpheres (CollisionDetection.cpp:27-48).  margin (optional):
// receives the signed gap the decision was taken on (< 0: contact).
template <class T>
GR_D CInfo<T> cp_spheres(T rA, T rB, const Tr<T>& a2w, const Tr<T>& b2w, T* margin = nullptr) {
  V3<T> cenA = a2w.o;
  V3<T> vecBA = b2w.o - cenA;
  T overlap = norm(vecBA) - rA - rB;
  if (margin) *margin = overlap;
  vecBA = vecBA / norm(vecBA);
  if (overlap < T(0)) return {cenA + (rA + T(0.5) * overlap) * vecBA, overlap * vecBA, overlap};
  return no_contact<T>();
}

// closestPointsRectangle (CollisionDetection.cpp:54-90); A's support is the
// full shape.  margin (optional): the support point's signed distance from
// the plane (< 0: contact).
template <class T>
GR_D CInfo<T> cp_rectangle(const SupCtx<T>& A, const Tr<T>& a2w, const Tr<T>& b2w, T* margin = nullptr) {
  V3<T> rPt = b2w.o;
  V3<T> rNorm = {b2w.R.m[2], b2w.R.m[5], b2w.R.m[8]};
  rNorm = copysign(T(1), dot(rNorm, a2w.o - rPt)) * rNorm;
  V3<T> pointA = apply(a2w, support(A, vm(-rNorm, a2w.R)));
  const T gap = dot(rNorm, pointA - rPt);
  if (margin) *margin = gap;
  if (gap < T(0)) {
    V3<T> pointB = dot(rPt - pointA, rNorm) * rNorm + pointA;
    V3<T> cv = pointB - pointA;
    return {T(0.5) * (pointA + pointB), cv, -norm(cv)};
  }
  return no_contact<T>();
}

// Outcome flags of one pair (all in one word: stores to it on different
// paths stay stores to one address, so the struct stays in registers).
constexpr uint32_t kNpGjk = 1u;       // GJK ran
constexpr uint32_t kNpDeep = 2u;
constexpr uint32_t kNpBackup = 4u;
constexpr uint32_t kNpDeferred = 8u;  // screening pass: not decided there (no result)
constexpr uint32_t kNpNear = 16u;     // FP32: the contact decision lay within the rounding band
struct NpStats {
  uint32_t bits;
  int iters;
  GR_D bool gjk() const { return (bits & kNpGjk) != 0; }
  GR_D bool deep() const { return (bits & kNpDeep) != 0; }
  GR_D bool backup() const { return (bits & kNpBackup) != 0; }
  GR_D bool deferred() const { return (bits & kNpDeferred) != 0; }
  GR_D bool near() const { return (bits & kNpNear) != 0; }
};

// FP32-mixed contact decisions.  The FP32 geometry of a pair differs from
// the FP64 one by the rounding of the pair frame (2^-24 of the centre
// offset), of the FP32 rotations and of the log2-domain superquadric
// support, whose coordinates carry up to ~2e-6 relative error for
// directions near an axis (two log2 terms of up to ~23 cancel there).
// Every FP32 gap on which a contact is decided -- bounding spheres, sphere
// pairs, GJK's separation bound and its converged distance -- therefore lies
// within kNearRel32 * (R_A + R_B) of the FP64 one (the bound is checked on
// near-contact superquadric pairs by the tests, which measure the FP32 and
// FP64 distances of the same pairs).  A decision whose margin is inside that
// band is flagged `near` and left to the FP64 re-run, so FP32-mixed contact
// decisions equal FP64 ones.  FP64 has no band.
constexpr float kNearRel32 = 1.6e-5f;
template <class T> GR_D T near_band(T rsum) {
  if constexpr (sizeof(T) == 4) return T(kNearRel32) * rsum;
  return T(0);
}

// closestPointsRigidBodies (CollisionDetection.cpp:181-284).  Physics
// semantics run GJK on the crust cores (the commented intent of lines 231-236).
// SV selects the physics semantics (signed-volume GJK on the crust cores);
// !SV is REF_QUIRKS (Johnson's sub-algorithm on the full shapes).
// warm (physics semantics): asked for a first GJK direction in the world
// frame only when the pair reaches GJK (fetch returns false: none); dir_w
// (optional): receives the search's direction in the world frame when GJK
// ran and produced one (left alone otherwise).
struct NoWarm {
  template <class V>
  GR_D bool fetch(V&) const { return false; }
};
// PAIR (physics semantics): two lanes per pair, as gjk_sv<PAIR>.
template <class T, bool SV, bool PAIR = false, class W = NoWarm>
GR_D CInfo<T> closest_points(const ShapeNP<T>& A, const ShapeNP<T>& B, const Tr<T>& a2w,
                             const Tr<T>& b2w, const GjkArgs& args, const T* verts_full,
                             const T* verts_core, NpStats& st, const W& warm = W(),
                             V3<T>* dir_w = nullptr) {
  constexpr bool quirks = !SV;
  const T band = near_band(A.rc + B.rc);  // 0 in FP64
  if ((A.kind == GRAINS_SPHERE && B.kind == GRAINS_SPHERE) || B.kind == GRAINS_RECTANGLE) {
    T margin;
    const CInfo<T> c = B.kind == GRAINS_RECTANGLE
                           ? cp_rectangle(sup_ctx(A, false, verts_full, verts_core), a2w, b2w, &margin)
                           : cp_spheres(A.rc, B.rc, a2w, b2w, &margin);
    if (band > T(0) && fabs(margin) <= band) st.bits |= kNpNear;
    return c;
  }
  T overlap = norm(b2w.o - a2w.o) - (A.rc + B.rc);
  // Bounding spheres apart by less than the band: FP64 may see them
  // overlap.  Physics semantics: the search runs anyway -- a separation it
  // proves beyond the band holds whichever way FP64 decides the spheres (no
  // contact either way), and any other outcome goes to the FP64 re-run,
  // which then starts from this search's direction; the reference semantics
  // leave such pairs to the re-run at once.
  const bool sphere_near = band > T(0) && overlap >= T(0) && overlap <= band;
  if (sphere_near && !SV) {
    st.bits |= kNpNear;
    return no_contact<T>();
  }
  if (overlap < T(0) || sphere_near) {
    if (!obb_intersect(A.bbox, B.bbox, a2w, b2w)) {
      if (sphere_near) st.bits |= kNpNear;
      return no_contact<T>();
    }
    {
      SupCtx<T> ca = sup_ctx(A, !quirks, verts_full, verts_core);
      SupCtx<T> cb = sup_ctx(B, !quirks, verts_full, verts_core);
      const T ctSum = A.crust + B.crust;
      GjkOut<T> g;
      if constexpr (SV) {
        // a separation proven beyond the band holds in FP64 too
        V3<T> warm_w;
        if (warm.fetch(warm_w)) {
          const V3<T> wa = vm(warm_w, a2w.R);  // into A's frame
          g = gjk_sv<T, PAIR>(ca, cb, a2w, b2w, args, A.rc + B.rc, ctSum + band, &wa);
        } else {
          g = gjk_sv<T, PAIR>(ca, cb, a2w, b2w, args, A.rc + B.rc, ctSum + band);
        }
        if (dir_w && g.has_v) *dir_w = mv(a2w.R, g.vdir);
      } else {
        g = gjk_jh<T, PAIR>(ca, cb, a2w, b2w, args);
      }
      st.bits |= kNpGjk;
      st.iters = g.iters;
      st.bits |= g.backup ? kNpBackup : 0u;
      if (g.separated) return no_contact<T>();
      T distance = g.dist - ctSum;
      if (g.deep) distance = -ctSum;
      // the converged distance is an upper bound within rel * dist of the
      // true one (gap test), and within the band of FP64's
      if (band > T(0) && !g.deep) {
        const T rel = args.rel > 0 ? T(args.rel) : Eps<T>::LOW;
        if (fabs(distance) <= band + rel * g.dist) st.bits |= kNpNear;
      }
      if (distance > T(0)) return no_contact<T>();
      if (sphere_near) {
        // a contact by GJK behind a bounding-sphere test FP32 cannot decide
        st.bits |= kNpNear;
        return no_contact<T>();
      }
      V3<T> ptA = apply(a2w, g.pa);
      V3<T> ptB = apply(b2w, g.pb);
      CInfo<T> c;
      c.cp = (ptA + ptB) / T(2);
      V3<T> cv = ptA - ptB;
      if (g.deep) {
        st.bits |= kNpDeep;
        cv = a2w.o - b2w.o;
        c.cp = (a2w.o + b2w.o) / T(2);
      }
      cv = cv / norm(cv);
      cv = round_tol(cv, Eps<T>::MID);
      c.cv = (-distance) * cv;
      c.overlap = distance;
      return c;
    }
  }
  return no_contact<T>();
}

// What of a pair the bounding spheres, the OBB or GJK's first support pair
// settle (physics semantics): most pairs of a resting or loose packing, none
// in contact.  Returns kNpGjk or 0 for a settled pair, kNpDeferred for one
// left to closest_points, which repeats it from the start with the same
// arithmetic (closest_points and gjk_sv up to the first separation test), so
// exactly the pairs it separates there are settled here.  warm_w: the first
// direction, in the world frame (zero or not finite: the centre difference);
// dir_w receives the direction of a pair GJK separates.
template <class T>
GR_D uint32_t screen_pair(const ShapeNP<T>& A, const ShapeNP<T>& B, const Tr<T>& a2w, const Tr<T>& b2w,
                          const T* verts_full, const T* verts_core, V3<T> warm_w, V3<T>& dir_w) {
  if ((A.kind == GRAINS_SPHERE && B.kind == GRAINS_SPHERE) || B.kind == GRAINS_RECTANGLE) return kNpDeferred;
  const T rsum = A.rc + B.rc;
  const T band = near_band(rsum);  // 0 in FP64
  const T overlap = norm(b2w.o - a2w.o) - rsum;
  const bool sphere_near = band > T(0) && overlap >= T(0) && overlap <= band;
  if (!(overlap < T(0) || sphere_near)) return 0u;
  if (!obb_intersect(A.bbox, B.bbox, a2w, b2w)) return sphere_near ? kNpDeferred : 0u;
  SupCtx<T> ca = sup_ctx(A, true, verts_full, verts_core);
  SupCtx<T> cb = sup_ctx(B, true, verts_full, verts_core);
  const T ctSum = A.crust + B.crust;
  Tr<T> b2a = relative(a2w, b2w);
  int ex;
  frexp(rsum, &ex);
  const T sc = ldexp(T(1), -ex);
  b2a.o = sc * b2a.o;
  const T sep_s = sc * (ctSum + band);
  const T nn = dot(warm_w, warm_w);
  const bool warm = nn > T(0) && nn < T(INFINITY);
  const V3<T> wa = vm(warm_w, a2w.R), v = -b2a.o;  // into A's frame
  const V3<T> dir = {warm ? wa.x : v.x, warm ? wa.y : v.y, warm ? wa.z : v.z};
  const T nd = norm(dir);
  if (!warm && !(nd > Eps<T>::HIGH)) return kNpDeferred;
  const V3<T> w = sc * support(ca, -dir) - apply(b2a, sc * support(cb, vm(dir, b2a.R)));
  const T lb = dot(dir, w) / nd;
  T mu = T(0);
  if (mu < lb) mu = lb;
  if (!(mu > sep_s)) return kNpDeferred;
  if (nd > T(0)) dir_w = mv(a2w.R, dir);
  return kNpGjk;
}

// The same under the reference semantics: the bounding spheres and the OBB
// (closest_points<T, false> up to its search).
template <class T>
GR_D uint32_t screen_ref(const ShapeNP<T>& A, const ShapeNP<T>& B, const Tr<T>& a2w, const Tr<T>& b2w) {
  if ((A.kind == GRAINS_SPHERE && B.kind == GRAINS_SPHERE) || B.kind == GRAINS_RECTANGLE) return kNpDeferred;
  const T rsum = A.rc + B.rc, band = near_band(rsum);  // 0 in FP64
  const T overlap = norm(b2w.o - a2w.o) - rsum;
  if (band > T(0) && overlap >= T(0) && overlap <= band) return kNpDeferred;
  return overlap < T(0) && obb_intersect(A.bbox, B.bbox, a2w, b2w) ? kNpDeferred : 0u;
}

// Hooke::performForcesCalculus + computeForces (HookeContactForceModel.cpp:91-186).
// Returns the force on A; `lever` = contact point - A's origin.
template <class T>
GR_D void hooke(const HookeP<T>& h, const CInfo<T>& ci, V3<T> relVel, V3<T> relAngVel, T m1, T m2,
                V3<T> lever, V3<T>& F, V3<T>& M) {
  V3<T> pen = ci.cv;
  V3<T> delFN = h.kn * pen;
  pen = pen / norm(pen);
  pen = round_tol(pen, Eps<T>::MID);
  V3<T> v_n = dot(relVel, pen) * pen;
  V3<T> v_t = relVel - v_n;
  T normv_t = norm(v_t);
  V3<T> tangent = {T(0), T(0), T(0)};
  if (normv_t > Eps<T>::MID) tangent = v_t / normv_t;
  T avmass = m1 * m2 / (m1 + m2);
  T omega0 = sqrt(h.kn / avmass);
  if (avmass == T(0)) {
    avmass = m2 == T(0) ? T(0.5) * m1 : T(0.5) * m2;
    omega0 = T(2) * sqrt(h.kn / avmass);
  }
  T muen = -omega0 * h.muen;
  delFN = delFN + (-T(2) * muen * avmass) * v_n;
  T normFN = norm(delFN);
  V3<T> delFT = (-h.etat * T(2) * avmass) * v_t;
  T fn = h.muc * normFN;
  T ft = norm(delFT);
  if (fn < ft) delFT = (-fn) * tangent;
  F = delFN + delFT;
  M = cross(lever, F);
  if (h.kr != T(0)) {
    V3<T> wn = dot(relAngVel, pen) * pen;
    V3<T> wt = relAngVel - wn;
    T normwt = norm(wt);
    V3<T> delM = (-h.kr * normFN * T(0.001)) * wn;
    if (normwt > Eps<T>::MID) delM = delM - (h.kr * normFN) * wt;
    M = M + delM;
  }
}

}  // namespace gr
