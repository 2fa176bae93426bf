// gr_capi.hip -- the C-ABI of include/grains_hip.h: scene set-up on the host
// (mass properties, linked-cell layout), device memory, and the step
// pipeline.  Replaces ComponentManagerGPU (Grains/Component/src/
// ComponentManagerGPU.cpp) and the GrainsGPU driver loop
// (Grains/Base/src/GrainsGPU.cpp:90-163).
#include <algorithm>
#include <cstdlib>
#include <cmath>
#include <cstdio>
#include <cstring>
#include <string>
#include <limits>
#include <memory>
#include <mutex>
#include <thread>
#include <vector>

#include "../../include/grains_hip.h"
#include "gr_internal.hpp"

using namespace gr;

namespace {

constexpr double kPi = 3.1415926535897932385;
constexpr double kEps = 1.e-10;

// ---- host mass properties (RigidBody ctor, RigidBody.cpp:19-59) -------------
struct HostShape {
  grains_shape_t s;
  double volume = 0, mass = 0, inertia[6] = {0}, inv[6] = {0};
  double rc = 0, rc_exact = 0, bbox[3] = {0}, core[5] = {0};
  double bbox_exact[3] = {0};  // OBB half-extents containing the shape (physics semantics)
  double gd[5] = {0};          // dims the support map reads (CYLINDER r, h/2; CONE r, h/4, sin)
  std::vector<double> verts, core_verts;
};

double beta_fn(double x, double y) { return std::exp(std::lgamma(x) + std::lgamma(y) - std::lgamma(x + y)); }

// Superquadric::computeCircumscribedRadius (Superquadric.cpp:122-155)
double sq_rc_reference(double a, double b, double c, double n1, double n2) {
  if (n1 == 2.0 && n2 == 2.0) return std::max(a, std::max(b, c));
  if (n1 == 2.0) {
    double al = std::pow(b / a, 2.0 / (n2 - 2.0));
    double xt = 1.0 / std::pow(1.0 + std::pow(al, n2), 1.0 / n2);
    return std::max(c, std::sqrt(a * xt * a * xt + al * b * xt * al * b * xt));
  }
  if (n2 == 2.0) {
    double m = std::max(a, b);
    double be = std::pow(c * c / (m * m), 1.0 / (n1 - 2.0));
    double xt = 1.0 / std::pow(1.0 + std::pow(be, n1), 1.0 / n1);
    return std::sqrt(m * xt * m * xt + be * c * xt * be * c * xt);
  }
  double al = std::pow(b / a, 2.0 / (n2 - 2.0));
  double ga = std::pow(1.0 + std::pow(al, n2), n1 / n2 - 1.0);
  double be = std::pow(ga * c * c / (a * a), 1.0 / (n1 - 1.0));
  double xt = 1.0 / std::pow(std::pow(1.0 + std::pow(al, n2), n1 / n2) + std::pow(be, n1), 1.0 / n1);
  return std::sqrt(a * xt * a * xt + al * b * xt * al * b * xt + be * c * xt * be * c * xt);
}

// True circumscribed radius: largest |p| over the critical points of every
// coordinate family of (|x/a|^n2 + |y/b|^n2)^(n1/n2) + |z/c|^n1 = 1.
double planar_max(double a, double b, double n) {
  double r = std::max(a, b);
  if (n > 2.0) {
    double t = std::pow(b / a, n / (n - 2.0));
    double x = a * std::pow(1.0 + std::pow(t * a / b, n), -1.0 / n);
    double c = std::sqrt(x * x + t * x * t * x);
    if (std::isfinite(c)) r = std::max(r, c);  // overflow near n = 2: the axis value is the limit
  }
  return r;
}
double sq_rc_exact(double a, double b, double c, double n1, double n2) {
  double r = std::max(planar_max(a, b, n2), std::max(planar_max(a, c, n1), planar_max(b, c, n1)));
  if (n1 > 2.0 && n2 > 2.0) {
    double al = std::pow(b / a, 2.0 / (n2 - 2.0));
    double T = 1.0 + std::pow(al, n2);
    double be = std::pow(c * c / (a * a) * std::pow(T, n1 / n2 - 1.0), 1.0 / (n1 - 2.0));
    double xt = std::pow(std::pow(T, n1 / n2) + std::pow(be, n1), -1.0 / n1);
    double x = a * xt, y = al * b * xt, z = be * c * xt;
    double q = std::sqrt(x * x + y * y + z * z);
    if (std::isfinite(q)) r = std::max(r, q);
  }
  return r;
}

// Convex hull volume, centroid and inertia (unit density, about the
// centroid): supporting planes through three points are facets, their
// coplanar points fan-triangulated around the facet centre.
void hull_mass(const std::vector<double>& P, double& vol, double* I6) {
  const int n = (int)P.size() / 3;
  auto pt = [&](int i) { return V3<double>{P[3 * i], P[3 * i + 1], P[3 * i + 2]}; };
  double V0 = 0, c[3] = {0, 0, 0}, acc[6] = {0, 0, 0, 0, 0, 0};
  for (int i = 0; i < n; ++i)
    for (int j = i + 1; j < n; ++j)
      for (int k = j + 1; k < n; ++k) {
        V3<double> a = pt(i), b = pt(j), cc = pt(k);
        V3<double> nr = cross(b - a, cc - a);
        double nn = norm(nr);
        if (nn == 0.0) continue;
        int pos = 0, neg = 0;
        bool first = true;
        std::vector<int> on;
        for (int l = 0; l < n; ++l) {
          double sd = dot(nr, pt(l) - a);
          if (sd > 1e-12 * nn) ++pos;
          else if (sd < -1e-12 * nn) ++neg;
          else {
            on.push_back(l);
            if (l < k && l != i && l != j) first = false;
          }
        }
        if ((pos && neg) || !first) continue;
        V3<double> out = pos ? -nr : nr;
        V3<double> ctr = {0, 0, 0};
        for (int l : on) ctr = ctr + pt(l);
        ctr = (1.0 / on.size()) * ctr;
        V3<double> e1 = a - ctr;
        e1 = (1.0 / norm(e1)) * e1;
        V3<double> e2 = cross((1.0 / nn) * out, e1);
        std::vector<std::pair<double, int>> ang;
        for (int l : on) {
          V3<double> dd = pt(l) - ctr;
          ang.push_back({std::atan2(dot(dd, e2), dot(dd, e1)), l});
        }
        std::sort(ang.begin(), ang.end());
        for (size_t t = 1; t + 1 < ang.size(); ++t) {
          V3<double> p0 = pt(ang[0].second), p1 = pt(ang[t].second), p2 = pt(ang[t + 1].second);
          double dv = dot(p0, cross(p1, p2)) / 6.0;
          V0 += dv;
          const double Q[3][3] = {{p0.x, p0.y, p0.z}, {p1.x, p1.y, p1.z}, {p2.x, p2.y, p2.z}};
          for (int q = 0; q < 3; ++q) c[q] += dv * (Q[0][q] + Q[1][q] + Q[2][q]) / 4.0;
          const int ii[6] = {0, 1, 2, 0, 0, 1}, jj[6] = {0, 1, 2, 1, 2, 2};
          for (int q = 0; q < 6; ++q) {
            double s1 = 0, si = 0, sj = 0;
            for (int r = 0; r < 3; ++r) {
              s1 += Q[r][ii[q]] * Q[r][jj[q]];
              si += Q[r][ii[q]];
              sj += Q[r][jj[q]];
            }
            acc[q] += dv / 20.0 * (s1 + si * sj);
          }
        }
      }
  vol = V0;
  for (int q = 0; q < 3; ++q) c[q] /= V0;
  double Sxx = acc[0] - V0 * c[0] * c[0], Syy = acc[1] - V0 * c[1] * c[1], Szz = acc[2] - V0 * c[2] * c[2];
  double Sxy = acc[3] - V0 * c[0] * c[1], Sxz = acc[4] - V0 * c[0] * c[2], Syz = acc[5] - V0 * c[1] * c[2];
  I6[0] = Syy + Szz;
  I6[1] = -Sxy;
  I6[2] = -Sxz;
  I6[3] = Sxx + Szz;
  I6[4] = -Syz;
  I6[5] = Sxx + Syy;
}

void sym_inv(const double* I, double* r) {
  double a = I[0], b = I[1], c = I[2], d = I[3], e = I[4], f = I[5];
  double A = d * f - e * e, B = -(b * f - c * e), C = b * e - c * d;
  double det = a * A + b * B + c * C;
  r[0] = A / det;
  r[1] = B / det;
  r[2] = C / det;
  r[3] = (a * f - c * c) / det;
  r[4] = -(a * e - b * c) / det;
  r[5] = (a * d - b * b) / det;
}

// Cone(r, h) members (Cone.cpp:9-14): r, h/4 and the sine of the half angle
void cone_dims(double* g, double r, double q) {
  g[0] = r;
  g[1] = q;
  g[2] = r / std::sqrt(r * r + 16.0 * q * q);
}

int derive_shape(HostShape& h, const grains_shape_t& s, const double* verts, uint32_t nverts) {
  h.s = s;
  const double* d = s.dims;
  double I[6] = {0, 0, 0, 0, 0, 0}, Ii[6] = {0, 0, 0, 0, 0, 0};
  switch (s.kind) {
    case GRAINS_SPHERE: {  // Sphere.cpp:72-105
      double r = d[0];
      if (!(r > 0)) return GRAINS_EINVAL;
      h.volume = 4.0 * kPi * r * r * r / 3.0;
      double r5 = r * r * r * r * r;
      I[5] = I[3] = I[0] = 8.0 * kPi / 15.0 * r5;
      Ii[5] = Ii[3] = Ii[0] = 1.0 / I[0];
      h.rc = r;
      h.bbox[0] = h.bbox[1] = h.bbox[2] = r;
      break;
    }
    case GRAINS_BOX: {  // Box.cpp:81-123
      double ex = d[0], ey = d[1], ez = d[2];
      if (!(ex > 0 && ey > 0 && ez > 0)) return GRAINS_EINVAL;
      h.volume = 8.0 * ex * ey * ez;
      I[0] = 8.0 * ex * ey * ez * (ey * ey + ez * ez) / 3.0;
      I[3] = 8.0 * ex * ey * ez * (ex * ex + ez * ez) / 3.0;
      I[5] = 8.0 * ex * ey * ez * (ey * ey + ex * ex) / 3.0;
      Ii[0] = 1.0 / I[0];
      Ii[3] = 1.0 / I[3];
      Ii[5] = 1.0 / I[5];
      h.rc = std::sqrt(ex * ex + ey * ey + ez * ez);
      h.bbox[0] = ex, h.bbox[1] = ey, h.bbox[2] = ez;
      break;
    }
    case GRAINS_SUPERQUADRIC: {  // Superquadric.cpp:81-163
      double a = d[0], b = d[1], c = d[2], n1 = d[3], n2 = d[4];
      if (!(a > 0 && b > 0 && c > 0 && n1 >= 2 && n2 >= 2)) return GRAINS_EINVAL;
      double e1 = 2.0 / n1, e2 = 2.0 / n2;
      h.volume = 2.0 / 3.0 * a * b * c * e1 * e2 * beta_fn(e1, 0.5 * e1) * beta_fn(0.5 * e2, 0.5 * e2);
      double Ci = 0.4 * a * b * c * e1 * e2;
      double p1 = beta_fn(1.5 * e2, 0.5 * e2) * beta_fn(2.0 * e1, 0.5 * e1);
      double p2 = c * c * beta_fn(0.5 * e2, 0.5 * e2) * beta_fn(1.5 * e1, e1);
      I[0] = Ci * (b * b * p1 + p2);
      I[3] = Ci * (a * a * p1 + p2);
      I[5] = Ci * (a * a + b * b) * p1;
      Ii[0] = 1.0 / I[0];
      Ii[3] = 1.0 / I[3];
      Ii[5] = 1.0 / I[5];
      h.rc = sq_rc_reference(a, b, c, n1, n2);
      h.rc_exact = sq_rc_exact(a, b, c, n1, n2);
      h.bbox[0] = a, h.bbox[1] = b, h.bbox[2] = c;
      break;
    }
    case GRAINS_CYLINDER: {  // Cylinder.cpp:9-12,72-111; dims: radius, height
      double r = d[0], hh = d[1] / 2.0;
      if (!(r > 0 && hh > 0)) return GRAINS_EINVAL;
      h.volume = 2.0 * kPi * hh * r * r;
      double r2 = r * r, c = 0.5 * kPi * hh * r2;
      I[0] = I[5] = c * (4.0 * hh * hh / 3.0 + r2);
      I[3] = 2.0 * c * r2;
      Ii[5] = Ii[0] = 1.0 / I[0];
      Ii[3] = 1.0 / I[3];
      h.rc = std::sqrt(r * r + hh * hh);
      h.bbox[0] = r, h.bbox[1] = hh, h.bbox[2] = r;
      break;
    }
    case GRAINS_CONE: {  // Cone.cpp:9-14,76-122; dims: base radius, height
      // origin at the centroid: apex at +3h/4 on y, base at -h/4
      double r = d[0], q = d[1] / 4.0;
      if (!(r > 0 && q > 0)) return GRAINS_EINVAL;
      h.volume = 4.0 * q * kPi * r * r / 3.0;
      double r2 = r * r, c = 0.2 * kPi * q * r2;
      I[0] = I[5] = c * (4.0 * q * q + r2);
      I[3] = 2.0 * c * r2;
      Ii[5] = Ii[0] = 1.0 / I[0];
      Ii[3] = 1.0 / I[3];
      h.rc = std::max(std::sqrt(r * r + q * q), 3.0 * q);
      // the reference box is centred on the centroid and leaves out the apex
      // region y in (h/2, 3h/4] (Cone.cpp:116-122)
      h.bbox[0] = r, h.bbox[1] = 2.0 * q, h.bbox[2] = r;
      break;
    }
    case GRAINS_RECTANGLE: {  // Rectangle.cpp:72-109
      double LX = d[0], LY = d[1];
      h.volume = 4.0 * LX * LY;
      I[0] = 4.0 / 3.0 * LX * LY * LY * LY;
      I[3] = 4.0 / 3.0 * LX * LX * LX * LY;
      I[5] = 2.0 / 3.0 * LX * LY * (LX * LX + LY * LY);
      Ii[0] = 1.0 / I[0];
      Ii[3] = 1.0 / I[3];
      Ii[5] = 1.0 / I[5];
      h.rc = std::sqrt(LX * LX + LY * LY);
      h.bbox[0] = LX, h.bbox[1] = LY, h.bbox[2] = 0.0;
      break;
    }
    case GRAINS_POLYHEDRON: {
      if (!verts || s.n_vertices < 4 || s.vertex_offset < 0 ||
          (uint64_t)s.vertex_offset + (uint64_t)s.n_vertices > nverts)
        return GRAINS_EINVAL;
      h.verts.assign(verts + 3 * (size_t)s.vertex_offset, verts + 3 * (size_t)(s.vertex_offset + s.n_vertices));
      hull_mass(h.verts, h.volume, I);
      if (!(h.volume > 0)) return GRAINS_EINVAL;
      sym_inv(I, Ii);
      for (int v = 0; v < s.n_vertices; ++v) {
        V3<double> p = {h.verts[3 * v], h.verts[3 * v + 1], h.verts[3 * v + 2]};
        h.rc = std::max(h.rc, norm(p));
        h.bbox[0] = std::max(h.bbox[0], std::fabs(p.x));
        h.bbox[1] = std::max(h.bbox[1], std::fabs(p.y));
        h.bbox[2] = std::max(h.bbox[2], std::fabs(p.z));
      }
      break;
    }
    default:
      return GRAINS_EUNSUPPORTED;
  }
  if (s.kind != GRAINS_SUPERQUADRIC) h.rc_exact = h.rc;
  for (int k = 0; k < 3; ++k) h.bbox_exact[k] = h.bbox[k];
  if (s.kind == GRAINS_CONE) h.bbox_exact[1] = 3.0 * d[1] / 4.0;
  std::copy(d, d + 5, h.gd);
  if (s.kind == GRAINS_CYLINDER) h.gd[1] = d[1] / 2.0;
  if (s.kind == GRAINS_CONE) cone_dims(h.gd, d[0], d[1] / 4.0);
  h.mass = s.density * h.volume;
  for (int i = 0; i < 6; ++i) {
    h.inertia[i] = s.density == 0 ? 0.0 : I[i] * s.density;
    h.inv[i] = s.density == 0 ? 0.0 : Ii[i] / s.density;
  }
  // crust core: RigidBody::m_scaling (RigidBody.cpp:27-31)
  std::copy(h.gd, h.gd + 5, h.core);
  switch (s.kind) {
    case GRAINS_SPHERE: h.core[0] = d[0] - s.crust; break;
    case GRAINS_CYLINDER:  // Cylinder(r - ct, h - 2 ct)
      h.core[0] = h.gd[0] - s.crust;
      h.core[1] = h.gd[1] - s.crust;
      break;
    case GRAINS_CONE:  // Cone(r - ct, h - 2 ct): y scaled by (h/2 - ct)/(h/2) about the centroid
      cone_dims(h.core, h.gd[0] - s.crust, h.gd[1] - 0.5 * s.crust);
      break;
    case GRAINS_BOX:
    case GRAINS_SUPERQUADRIC:
      for (int k = 0; k < 3; ++k) h.core[k] = d[k] - s.crust;
      break;
    case GRAINS_POLYHEDRON:
      h.core_verts = h.verts;
      for (size_t v = 0; v < h.verts.size(); ++v) {
        int k = v % 3;
        h.core_verts[v] *= h.bbox[k] > 0 ? (h.bbox[k] - s.crust) / h.bbox[k] : 1.0;
      }
      break;
    default: break;
  }
  return GRAINS_OK;
}

template <class T>
ShapeNP<T> to_np(const HostShape& h, bool quirks, int32_t voff) {
  ShapeNP<T> r;
  std::memset(&r, 0, sizeof(r));
  r.kind = h.s.kind;
  r.material = h.s.material;
  r.nv = h.s.n_vertices;
  r.voff = voff;
  for (int k = 0; k < 5; ++k) {
    r.dims[k] = T(h.gd[k]);
    r.core[k] = T(h.core[k]);
  }
  r.crust = T(h.s.crust);
  r.rc = T(quirks ? h.rc : h.rc_exact);
  for (int k = 0; k < 3; ++k) r.bbox[k] = T(quirks ? h.bbox[k] : h.bbox_exact[k]);
  r.mass = T(h.mass);
  r.rc_max = T(std::max(h.rc, h.rc_exact));
  return r;
}

}  // namespace

// ---- context ------------------------------------------------------------------
struct grains_ctx {
  grains_config_t cfg;
  std::string err;
  hipStream_t stream = nullptr;
  hipEvent_t ev0 = nullptr, ev1 = nullptr;
  // the second stream of a step (the integration of the particles the
  // narrow screen settled, beside the rest of the narrow phase), its events
  hipStream_t side = nullptr;
  hipEvent_t ev_fork = nullptr, ev_join = nullptr;
  std::vector<HostShape> shapes;
  std::vector<double> verts_in;
  std::vector<grains_hooke_t> tables;
  uint32_t nmat = 0, ntables = 0;
  std::vector<grains_sim_t> sims;
  std::vector<uint32_t> obs_shape, obs_sim;
  std::vector<double> obs_tr;
  std::vector<uint32_t> pshape, psim;
  uint64_t n = 0;
  bool layout_ok = false;
  DevScene d;
  std::vector<void*> allocs;       // layout-dependent buffers
  std::vector<void*> state_allocs; // particle state
  int passes = 1;      // LSD radix passes of the cell keys
  int digit_bits = 8;  // bits per pass
  int ref_passes = 1;  // passes the reference's cell keys take (grains_stats_t.sort_passes), and their digits
  int ref_digit_bits = 8;
  uint32_t *keys_s = nullptr, *idx_s = nullptr;
  hipGraph_t graph = nullptr;            // one step
  hipGraphExec_t graph_exec = nullptr;
  hipGraph_t graph_multi = nullptr;      // graph_steps steps
  hipGraphExec_t graph_multi_exec = nullptr;
  uint32_t graph_steps = 1;
  hipGraph_t graph_build = nullptr;      // the neighbour lists' build
  hipGraphExec_t graph_build_exec = nullptr;
  grains_stats_t stats;
  std::vector<SimGrid> grids;   // the reference's cells
  std::vector<SimGrid> sgrids;  // the search's
  // Neighbour lists.  They stand from one call to the next while nothing but
  // the steps themselves moves the particles; lists_ok is cleared wherever
  // the state or the layout is set.
  bool lists_ok = false;
  bool skin_back = false;       // without a skin for one step: its centres lie outside a periodic side
  uint32_t since_build = 0;     // steps taken since they were built
  uint32_t interval = 8;        // steps they are expected to hold, and whether a build has shown it
  bool interval_known = false;
  unsigned char* host_words = nullptr;  // pinned: the counters and the list words, read back together
  // grains_get_state: rows of up to rows_cap particles in pinned memory, two
  // of them when the state takes several (the events are the context's GPU's,
  // whichever is current when the state is read)
  std::mutex rows_mu;
  double* rows[2] = {nullptr, nullptr};
  hipEvent_t rows_ev[2] = {nullptr, nullptr};
  uint64_t rows_cap = 0;
  // profiling: events around the phases of each step
  bool profiling = false;
  bool capturing = false;
  std::vector<hipEvent_t> pev;
  uint32_t pev_used = 0;
  double phase_ms[GRAINS_NUM_PHASES] = {0};
  // differentiation: the recorded trajectory and the sweep's buffers
  bool adj_rec = false;
  uint32_t adj_every = 0;
  uint64_t adj_steps = 0;
  std::vector<void*> adj_cp;      // state every adj_every steps (13 planes)
  std::vector<void*> adj_allocs;  // sweep buffers
  uint64_t adj_cap = 0;           // the most device bytes the recording and its sweeps hold (0: what the device has)
  std::vector<void*> adj_gjk;     // the searches' records
  std::vector<double*> adj_log;   // per block of adj_every steps, the states between (null: run again from its checkpoint)
  std::vector<void*> adj_log_allocs;
  bool adj_log_off = false;       // it gave way to what the recording and the sweep cannot do without
  bool adj_log_ok = false;        // the logged steps followed each other (no state set between)
  AdjBufs ab{};
  double *adj_blk = nullptr, *adj_save = nullptr;
  int32_t* adj_count = nullptr;
  // grains_gjk_batch_device_noalloc: the device address of `scratch` on this
  // context's GPU, and the shape tables it copies there, built by
  // grains_set_shapes (ShapeNP<double>, ShapeNP<float>, vertices FP64, FP32)
  unsigned char* scratch = nullptr;
  std::vector<ShapeNP<double>> na_np64;
  std::vector<ShapeNP<float>> na_np32;
  std::vector<double> na_v64;
  std::vector<float> na_v32;
};

static void free_rows(grains_ctx* ctx);
#define GR_HIP(call)                                                                    \
  do {                                                                                  \
    hipError_t e_ = (call);                                                             \
    if (e_ != hipSuccess) {                                                             \
      ctx->err = std::string(#call) + ": " + hipGetErrorString(e_);                     \
      return GRAINS_EDEVICE;                                                            \
    }                                                                                   \
  } while (0)

static int fail(grains_ctx* ctx, int code, const std::string& msg) {
  ctx->err = msg;
  return code;
}

template <class P>
static int dalloc(grains_ctx* ctx, P** p, size_t bytes, std::vector<void*>& list) {
  void* q = nullptr;
  if (bytes == 0) bytes = 16;
  hipError_t e = hipMalloc(&q, bytes);
  if (e != hipSuccess) {
    (void)hipGetLastError();
    return fail(ctx, GRAINS_ENOMEM, "hipMalloc of " + std::to_string(bytes) + " bytes failed");
  }
  list.push_back(q);
  *p = (P*)q;
  return GRAINS_OK;
}

static void free_list(std::vector<void*>& list) {
  for (void* p : list) (void)hipFree(p);
  list.clear();
}

static void free_events(grains_ctx* ctx) {
  for (hipEvent_t e : ctx->pev) (void)hipEventDestroy(e);
  ctx->pev.clear();
}

static void adj_drop(grains_ctx* ctx);

// candidate search mode: staging the neighbour windows in LDS pays off when
// cells hold many particles (measured: 250k polyhedra at ~145 per cell, 20 %
// faster; superquadric beds at ~6 per cell, 40 % slower)
// mode 0: the half-shell search where it applies (it shares dense cells
// among several groups), else the staged search when particles outnumber
// cells 8 to 1
static int32_t staging_of(int32_t mode, uint64_t n, uint64_t ncells, int32_t half) {
  if (mode == 0) return !half && n > 8 * ncells ? 1 : 0;
  return mode == 2 ? 1 : 0;
}

// the half-shell direct search: asked for (modes 0 and 1), and every
// periodic axis of every sim has at least three cells (with fewer, a
// neighbour cell is both a forward and a backward one)
static int32_t half_of(int32_t mode, const std::vector<SimGrid>& grids) {
  if (mode == 2 || mode == 3) return 0;
  for (const SimGrid& g : grids)
    for (int k = 0; k < 3; ++k)
      if (((g.periodic >> k) & 1) && g.n3[k] < 3) return 0;
  return 1;
}

static void drop_graph(grains_ctx* ctx) {
  if (ctx->graph_exec) (void)hipGraphExecDestroy(ctx->graph_exec);
  if (ctx->graph) (void)hipGraphDestroy(ctx->graph);
  if (ctx->graph_multi_exec) (void)hipGraphExecDestroy(ctx->graph_multi_exec);
  if (ctx->graph_multi) (void)hipGraphDestroy(ctx->graph_multi);
  ctx->graph_exec = nullptr;
  ctx->graph = nullptr;
  if (ctx->graph_build_exec) (void)hipGraphExecDestroy(ctx->graph_build_exec);
  if (ctx->graph_build) (void)hipGraphDestroy(ctx->graph_build);
  ctx->graph_multi_exec = nullptr;
  ctx->graph_multi = nullptr;
  ctx->graph_build_exec = nullptr;
  ctx->graph_build = nullptr;
}

constexpr size_t kCounterBytes = (size_t)kNumCounters * kCntSlots * 8;
constexpr size_t kWordBytes = kCounterBytes + kNlWords * 4;

extern "C" const char* grains_version(void) { return "grains_hip 0.1 gfx950"; }

// ---- the allocation-free GJK batch's device memory ------------------------------
// The shape tables of grains_gjk_batch_device_noalloc live in this
// file-scope array: every GPU the library runs on holds its own copy, at its
// own address, until the process ends.  Host code never passes the array's
// name to a kernel or a copy (on the host it names a stand-in, not device
// memory): grains_create looks up its device address once per GPU with
// hipGetSymbolAddress, with that GPU current, and every use goes through
// that address.
constexpr size_t kScratchBytes = size_t(1) << 20;
static __device__ __align__(256) unsigned char scratch[kScratchBytes];

constexpr int kMaxDevices = 64;
static std::mutex g_scratch_mu;
static unsigned char* g_scratch_addr[kMaxDevices] = {};

// The device address of `scratch` on the current GPU.
static int scratch_address(unsigned char** out) {
  int dev = -1;
  if (hipGetDevice(&dev) != hipSuccess || dev < 0 || dev >= kMaxDevices) {
    (void)hipGetLastError();
    return GRAINS_EDEVICE;
  }
  std::lock_guard<std::mutex> lock(g_scratch_mu);
  if (!g_scratch_addr[dev]) {
    void* p = nullptr;
    if (hipGetSymbolAddress(&p, HIP_SYMBOL(scratch)) != hipSuccess || !p) {
      (void)hipGetLastError();
      return GRAINS_EDEVICE;
    }
    g_scratch_addr[dev] = (unsigned char*)p;
  }
  *out = g_scratch_addr[dev];
  return GRAINS_OK;
}

extern "C" int grains_create(const grains_config_t* cfg, grains_ctx_t** out) {
  if (!cfg || !out) return GRAINS_EINVAL;
  *out = nullptr;
  if (!(cfg->dt > 0) || (cfg->precision != GRAINS_FP64 && cfg->precision != GRAINS_FP32_MIXED))
    return GRAINS_EINVAL;
  grains_ctx* ctx = new (std::nothrow) grains_ctx();
  if (!ctx) return GRAINS_ENOMEM;
  ctx->cfg = *cfg;
  if (ctx->cfg.max_neighbors <= 0) ctx->cfg.max_neighbors = 48;
  if (ctx->cfg.block_size <= 0) ctx->cfg.block_size = 256;
  if (ctx->cfg.block_size != 64 && ctx->cfg.block_size != 128 && ctx->cfg.block_size != 256) {
    delete ctx;
    return GRAINS_EINVAL;
  }
  if (ctx->cfg.gjk_rel_tol_fp64 < 0) {
    delete ctx;
    return GRAINS_EINVAL;
  }
  if (const char* e = std::getenv("GRAINS_ADJOINT_BYTES")) ctx->adj_cap = std::strtoull(e, nullptr, 10);
  if (ctx->cfg.gjk_rel_tol_fp64 == 0) ctx->cfg.gjk_rel_tol_fp64 = 1e-10;
  if (ctx->cfg.narrow_blocks_per_cu <= 0) ctx->cfg.narrow_blocks_per_cu = 8;
  // the narrow phase's queue segments and their scan are sized for at most
  // kMaxNarrowPerCu resident blocks per CU (finalize)
  if (ctx->cfg.narrow_blocks_per_cu > kMaxNarrowPerCu) {
    delete ctx;
    return GRAINS_EINVAL;
  }
  if (ctx->cfg.narrow_passes == 0) ctx->cfg.narrow_passes = 2;
  if (ctx->cfg.narrow_passes != 1 && ctx->cfg.narrow_passes != 2) {
    delete ctx;
    return GRAINS_EINVAL;
  }
  if (ctx->cfg.candidate_staging < 0 || ctx->cfg.candidate_staging > 3) {
    delete ctx;
    return GRAINS_EINVAL;
  }
  if (ctx->cfg.integrator < GRAINS_FIRST_ORDER_EXPLICIT || ctx->cfg.integrator > GRAINS_SECOND_ORDER_ADAMS_BASHFORTH) {
    delete ctx;
    return GRAINS_EINVAL;
  }
  std::memset(&ctx->stats, 0, sizeof(ctx->stats));
  std::memset(&ctx->d, 0, sizeof(ctx->d));
  int ndev = 0;
  if (hipGetDeviceCount(&ndev) != hipSuccess || ndev == 0) {
    (void)hipGetLastError();
    delete ctx;
    return GRAINS_EDEVICE;
  }
  if (hipStreamCreateWithFlags(&ctx->stream, hipStreamNonBlocking) != hipSuccess ||
      hipEventCreate(&ctx->ev0) != hipSuccess || hipEventCreate(&ctx->ev1) != hipSuccess ||
      hipStreamCreateWithFlags(&ctx->side, hipStreamNonBlocking) != hipSuccess ||
      hipEventCreateWithFlags(&ctx->ev_fork, hipEventDisableTiming) != hipSuccess ||
      hipEventCreateWithFlags(&ctx->ev_join, hipEventDisableTiming) != hipSuccess ||
      hipEventCreateWithFlags(&ctx->rows_ev[0], hipEventDisableTiming) != hipSuccess ||
      hipEventCreateWithFlags(&ctx->rows_ev[1], hipEventDisableTiming) != hipSuccess ||
      hipHostMalloc((void**)&ctx->host_words, kWordBytes, hipHostMallocDefault) != hipSuccess) {
    (void)hipGetLastError();
    grains_destroy(ctx);
    return GRAINS_EDEVICE;
  }
  if (int rc = scratch_address(&ctx->scratch)) {
    grains_destroy(ctx);
    return rc;
  }
  *out = ctx;
  return GRAINS_OK;
}

extern "C" void grains_destroy(grains_ctx_t* ctx) {
  if (!ctx) return;
  if (ctx->stream) (void)hipStreamSynchronize(ctx->stream);
  drop_graph(ctx);
  free_events(ctx);
  adj_drop(ctx);
  free_list(ctx->allocs);
  free_list(ctx->state_allocs);
  if (ctx->host_words) (void)hipHostFree(ctx->host_words);
  free_rows(ctx);
  if (ctx->ev0) (void)hipEventDestroy(ctx->ev0);
  if (ctx->ev1) (void)hipEventDestroy(ctx->ev1);
  if (ctx->ev_fork) (void)hipEventDestroy(ctx->ev_fork);
  if (ctx->ev_join) (void)hipEventDestroy(ctx->ev_join);
  for (hipEvent_t e : ctx->rows_ev)
    if (e) (void)hipEventDestroy(e);
  if (ctx->side) (void)hipStreamDestroy(ctx->side);
  if (ctx->stream) (void)hipStreamDestroy(ctx->stream);
  delete ctx;
}

extern "C" const char* grains_last_error(const grains_ctx_t* ctx) { return ctx ? ctx->err.c_str() : "null context"; }

// Shape tables of the GJK batches: the full shapes (no crust core), each
// polyhedron's vertices appended in shape order (one zero vertex when there
// are none, so the tables are never empty).
static void batch_tables(grains_ctx* ctx) {
  const size_t S = ctx->shapes.size();
  const bool quirks = (ctx->cfg.flags & GRAINS_REF_QUIRKS) != 0;
  ctx->na_np64.resize(S);
  ctx->na_np32.resize(S);
  ctx->na_v64.clear();
  for (size_t i = 0; i < S; ++i) {
    const int32_t voff = (int32_t)(ctx->na_v64.size() / 3);
    ctx->na_np64[i] = to_np<double>(ctx->shapes[i], quirks, voff);
    ctx->na_np32[i] = to_np<float>(ctx->shapes[i], quirks, voff);
    ctx->na_v64.insert(ctx->na_v64.end(), ctx->shapes[i].verts.begin(), ctx->shapes[i].verts.end());
  }
  if (ctx->na_v64.empty()) ctx->na_v64.assign(3, 0.0);
  ctx->na_v32.assign(ctx->na_v64.begin(), ctx->na_v64.end());
}

extern "C" int grains_set_shapes(grains_ctx_t* ctx, const grains_shape_t* shapes, uint32_t n_shapes,
                                 const double* vertices, uint32_t n_vertices) {
  if (!ctx || (!shapes && n_shapes)) return GRAINS_EINVAL;
  std::vector<HostShape> hs(n_shapes);
  for (uint32_t i = 0; i < n_shapes; ++i) {
    int rc = derive_shape(hs[i], shapes[i], vertices, n_vertices);
    if (rc) return fail(ctx, rc, "shape " + std::to_string(i) + " is invalid or unsupported");
  }
  ctx->shapes.swap(hs);
  ctx->verts_in.assign(vertices, vertices + 3 * (size_t)n_vertices);
  batch_tables(ctx);
  ctx->layout_ok = false;
  return GRAINS_OK;
}

extern "C" int grains_set_contact_tables(grains_ctx_t* ctx, const grains_hooke_t* t, uint32_t n_materials,
                                         uint32_t n_tables) {
  if (!ctx || !t || !n_materials || !n_tables) return GRAINS_EINVAL;
  const size_t per = (size_t)n_materials * (n_materials + 1) / 2;
  for (size_t i = 0; i < per * n_tables; ++i)
    if (!(t[i].kn > 0) || !(t[i].en > 0 && t[i].en <= 1))
      return fail(ctx, GRAINS_EINVAL, "contact table entry " + std::to_string(i) + ": need kn > 0, 0 < en <= 1");
  ctx->tables.assign(t, t + per * n_tables);
  ctx->nmat = n_materials;
  ctx->ntables = n_tables;
  ctx->layout_ok = false;
  return GRAINS_OK;
}

extern "C" int grains_set_sims(grains_ctx_t* ctx, const grains_sim_t* sims, uint32_t n_sims) {
  if (!ctx || !sims || !n_sims) return GRAINS_EINVAL;
  ctx->sims.assign(sims, sims + n_sims);
  ctx->layout_ok = false;
  return GRAINS_OK;
}

extern "C" int grains_set_obstacles(grains_ctx_t* ctx, const uint32_t* shape, const uint32_t* sim,
                                    const double* transforms, uint32_t n) {
  if (!ctx || (n && (!shape || !transforms))) return GRAINS_EINVAL;
  ctx->obs_shape.assign(shape, shape + n);
  ctx->obs_sim.assign(n, 0u);
  if (sim) ctx->obs_sim.assign(sim, sim + n);
  ctx->obs_tr.assign(transforms, transforms + 12 * (size_t)n);
  ctx->layout_ok = false;
  return GRAINS_OK;
}

// The schemes' history: NaN in every plane, so the next step is a first-order
// one (ADAMS_BASHFORTH) or a half kick (LEAPFROG).
static int hist_reset(grains_ctx* ctx) {
  if (!ctx->d.ab_hist) return GRAINS_OK;
  std::vector<double> nan(12 * ctx->n, std::numeric_limits<double>::quiet_NaN());
  GR_HIP(hipMemcpy(ctx->d.ab_hist, nan.data(), nan.size() * sizeof(double), hipMemcpyHostToDevice));
  return GRAINS_OK;
}

// A new state: the neighbour lists no longer hold, and the warm-start records
// are forgotten: the next step searches cold (it is not the continuation of
// the recorded directions).
static int warm_reset(grains_ctx* ctx) {
  ctx->lists_ok = false;
  ctx->adj_log_ok = false;
  if (!ctx->d.ws_nb) return GRAINS_OK;
  launch_fill_u32((uint32_t*)ctx->d.ws_nb, 4 * ctx->n, 0u, ctx->stream);
  GR_HIP(hipGetLastError());
  GR_HIP(hipStreamSynchronize(ctx->stream));
  return GRAINS_OK;
}

static int alloc_state(grains_ctx* ctx) {
  free_list(ctx->state_allocs);
  const uint64_t n = ctx->n;
  DevScene& d = ctx->d;
  auto& L = ctx->state_allocs;
  int rc;
  d.ab_hist = nullptr;
  if ((ctx->cfg.integrator == GRAINS_SECOND_ORDER_ADAMS_BASHFORTH ||
       ctx->cfg.integrator == GRAINS_SECOND_ORDER_LEAPFROG) &&
      ((rc = dalloc(ctx, &d.ab_hist, 12 * n * sizeof(double), L)) || (rc = hist_reset(ctx))))
    return rc;
  // the state's 13 planes in one block: copied at once (snapshots, checkpoints)
  if ((rc = dalloc(ctx, &d.pos, 13 * n * sizeof(double), L)) ||
      (rc = dalloc(ctx, &d.shape, n * sizeof(uint32_t), L)) || (rc = dalloc(ctx, &d.sim, n * sizeof(uint32_t), L)) ||
      (rc = dalloc(ctx, &d.contact_count, n * sizeof(int32_t), L)) ||
      (rc = dalloc(ctx, &d.last_force, 3 * n * sizeof(double), L)) ||
      (rc = dalloc(ctx, &d.last_torque, 3 * n * sizeof(double), L)))
    return rc;
  d.quat = d.pos + 3 * n;
  d.vel = d.pos + 7 * n;
  d.omega = d.pos + 10 * n;
  std::vector<double> zero(4 * n, 0.0), q(4 * n, 0.0);
  for (uint64_t i = 0; i < n; ++i) q[3 * n + i] = 1.0;
  GR_HIP(hipMemcpy(d.pos, zero.data(), 3 * n * sizeof(double), hipMemcpyHostToDevice));
  GR_HIP(hipMemcpy(d.vel, zero.data(), 3 * n * sizeof(double), hipMemcpyHostToDevice));
  GR_HIP(hipMemcpy(d.omega, zero.data(), 3 * n * sizeof(double), hipMemcpyHostToDevice));
  GR_HIP(hipMemcpy(d.last_force, zero.data(), 3 * n * sizeof(double), hipMemcpyHostToDevice));
  GR_HIP(hipMemcpy(d.last_torque, zero.data(), 3 * n * sizeof(double), hipMemcpyHostToDevice));
  GR_HIP(hipMemcpy(d.quat, q.data(), 4 * n * sizeof(double), hipMemcpyHostToDevice));
  GR_HIP(hipMemcpy(d.contact_count, zero.data(), n * sizeof(int32_t), hipMemcpyHostToDevice));
  GR_HIP(hipMemcpy(d.shape, ctx->pshape.data(), n * sizeof(uint32_t), hipMemcpyHostToDevice));
  GR_HIP(hipMemcpy(d.sim, ctx->psim.data(), n * sizeof(uint32_t), hipMemcpyHostToDevice));
  return GRAINS_OK;
}

extern "C" int grains_set_particles(grains_ctx_t* ctx, const uint32_t* shape, const uint32_t* sim, uint64_t n) {
  if (!ctx || !shape || !n) return GRAINS_EINVAL;
  if (n >= (1ull << 31)) return fail(ctx, GRAINS_EINVAL, "too many particles");
  if (ctx->shapes.empty() || ctx->sims.empty())
    return fail(ctx, GRAINS_ESTATE, "set shapes and sims before particles");
  for (uint64_t i = 0; i < n; ++i) {
    if (shape[i] >= ctx->shapes.size()) return fail(ctx, GRAINS_EINVAL, "particle shape index out of range");
    int k = ctx->shapes[shape[i]].s.kind;
    if (k == GRAINS_RECTANGLE) return fail(ctx, GRAINS_EINVAL, "a particle cannot be a Rectangle");
    if (ctx->shapes[shape[i]].mass <= 0) return fail(ctx, GRAINS_EINVAL, "particle mass must be > 0");
    uint32_t sm = sim ? sim[i] : 0u;
    if (sm >= ctx->sims.size()) return fail(ctx, GRAINS_EINVAL, "particle sim index out of range");
    if (i && sim && sim[i] < sim[i - 1]) return fail(ctx, GRAINS_EINVAL, "particles must be grouped by ascending sim");
  }
  ctx->n = n;
  ctx->pshape.assign(shape, shape + n);
  ctx->psim.assign(n, 0u);
  if (sim) ctx->psim.assign(sim, sim + n);
  ctx->d.n = n;
  ctx->layout_ok = false;
  drop_graph(ctx);
  free_list(ctx->allocs);
  return alloc_state(ctx);
}

// cell layout, obstacle ranges, shape tables and work buffers
// One of the screening pass's queues: the blocks on one of the kXcds dies
// share ecap / kXcds + 64 entries, in turns of a block's threads, and every
// kDeferQueues-th block fills the same queue.  For any launch shape the
// queues together hold at most (blocks + kDeferQueues - 1) ((ecap + 64 kXcds)
// / blocks + threads) words, which defer_words bounds (a launch has at least
// one block per CU and at most kMaxNarrowPerCu).
static void set_defer_cap(grains_ctx* ctx) {
  DevScene& d = ctx->d;
  const uint64_t per = (uint64_t)d.narrow_blocks * d.block;
  const uint64_t block_cap = ((d.ecap + 64 * kXcds + per - 1) / per) * d.block;
  d.defer_cap = (uint32_t)(block_cap * ((d.narrow_blocks + kDeferQueues - 1) / kDeferQueues));
}
static uint64_t defer_words(uint64_t ecap) {
  const uint64_t cus = (uint64_t)cu_count();
  return ecap + (kDeferQueues - 1) * (ecap / cus + 1) + (cus * kMaxNarrowPerCu + kDeferQueues) * 256 +
         64 * kXcds * kDeferQueues;
}

// Device memory of the recording and its sweeps, within adj_cap.
template <class P>
static int adj_spare(grains_ctx* ctx, P** p, size_t bytes, std::vector<void*>& list) {
  if (ctx->adj_cap) {
    uint64_t held = bytes;
    for (const auto* l : {&ctx->adj_cp, &ctx->adj_allocs, &ctx->adj_log_allocs, &ctx->adj_gjk})
      for (void* q : *l) {
        size_t b = 0;
        GR_HIP(hipMemPtrGetInfo(q, &b));
        held += b;
      }
    if (held > ctx->adj_cap)
      return fail(ctx, GRAINS_ENOMEM, std::to_string(bytes) + " bytes more for the adjoint pass GRAINS_ADJOINT_BYTES");
  }
  return dalloc(ctx, p, bytes, list);
}
// The same for what cannot be done without: what is only kept to spare work,
// the logged states and the searches' records, gives way to it.
template <class P>
static int adj_dalloc(grains_ctx* ctx, P** p, size_t bytes, std::vector<void*>& list) {
  const int rc = adj_spare(ctx, p, bytes, list);
  if (rc != GRAINS_ENOMEM || (ctx->adj_log_allocs.empty() && ctx->adj_gjk.empty())) return rc;
  launch_log_set(ctx->d, StateLog{}, 0u, ctx->stream);  // (set again before the next steps)
  GR_HIP(hipStreamSynchronize(ctx->stream));
  ctx->adj_log_off = true;
  ctx->adj_log.assign(ctx->adj_log.size(), nullptr);
  ctx->ab.gjk = nullptr;
  free_list(ctx->adj_log_allocs);
  free_list(ctx->adj_gjk);
  return adj_spare(ctx, p, bytes, list);
}

static void adj_drop(grains_ctx* ctx) {
  if (ctx->adj_rec) drop_graph(ctx);  // a recorded step logs its state
  free_list(ctx->adj_cp);
  free_list(ctx->adj_allocs);
  free_list(ctx->adj_gjk);
  free_list(ctx->adj_log_allocs);
  ctx->adj_log.clear();
  ctx->adj_rec = false;
  ctx->adj_steps = 0;
  ctx->ab = AdjBufs{};
  ctx->adj_blk = ctx->adj_save = nullptr;
  ctx->adj_count = nullptr;
}

// The search's cells, and how it runs over them: with a skin those of
// ctx->sgrids; without one the reference's (ctx->grids), every build for its
// step alone and a list the step's own candidates, so that it needs no more
// of max_neighbors than they do, whatever the cells' size.
static const std::vector<SimGrid>& search_grids(const grains_ctx* ctx) { return ctx->d.skin ? ctx->sgrids : ctx->grids; }
static void set_search(grains_ctx* ctx, bool skin) {
  DevScene& d = ctx->d;
  d.skin = skin ? 1 : 0;
  const std::vector<SimGrid>& grids = search_grids(ctx);
  const SimGrid& g = grids.back();
  d.ncells = g.base + (uint32_t)((uint64_t)g.n3[0] * g.n3[1] * g.n3[2]);
  int bits = 1;
  while (bits < 32 && (1ull << bits) < d.ncells) ++bits;
  // fewest LSD passes of digits up to kRadixMaxBits wide, digits at least 8
  // bits: an 18-bit key sorts in 2 passes of 9 bits instead of 3 of 8
  ctx->passes = (bits + kRadixMaxBits - 1) / kRadixMaxBits;
  ctx->digit_bits = std::max(8, (bits + ctx->passes - 1) / ctx->passes);
  d.cand_half = half_of(ctx->cfg.candidate_staging, grids);
  d.cand_staged = staging_of(ctx->cfg.candidate_staging, ctx->n, d.ncells, d.cand_half);
  // dense cells on average: the half-shell search takes its groups (several
  // on a dense cell) from a work list built each step
  d.half_wl = ctx->n > 8 * (uint64_t)d.ncells ? 1 : 0;
}

static int finalize(grains_ctx* ctx) {
  if (ctx->layout_ok) return GRAINS_OK;
  if (!ctx->n) return fail(ctx, GRAINS_ESTATE, "no particles");
  if (ctx->tables.empty()) return fail(ctx, GRAINS_ESTATE, "no contact table");
  drop_graph(ctx);
  adj_drop(ctx);  // a new layout ends a recorded trajectory
  free_list(ctx->allocs);
  DevScene& d = ctx->d;
  const bool quirks = (ctx->cfg.flags & GRAINS_REF_QUIRKS) != 0;
  const uint32_t ns = (uint32_t)ctx->sims.size();
  d.balls = 1;
  for (uint32_t k : ctx->pshape)
    if (ctx->shapes[k].s.kind != GRAINS_SPHERE) {
      d.balls = 0;
      break;
    }
  d.gen_obs = 0;
  for (uint32_t s : ctx->obs_shape) {
    if (s >= ctx->shapes.size()) return fail(ctx, GRAINS_EINVAL, "obstacle shape index out of range");
    if (ctx->shapes[s].s.kind != GRAINS_RECTANGLE) d.gen_obs = 1;
  }
  for (uint32_t s : ctx->obs_sim)
    if (s >= ns) return fail(ctx, GRAINS_EINVAL, "obstacle sim index out of range");
  for (const auto& h : ctx->shapes)
    if ((uint32_t)h.s.material >= ctx->nmat) return fail(ctx, GRAINS_EINVAL, "material id beyond the contact table");
  // obstacles grouped by sim (stable, so their order within a sim is kept)
  std::vector<uint32_t> ord(ctx->obs_shape.size());
  for (size_t i = 0; i < ord.size(); ++i) ord[i] = (uint32_t)i;
  std::stable_sort(ord.begin(), ord.end(), [&](uint32_t a, uint32_t b) { return ctx->obs_sim[a] < ctx->obs_sim[b]; });
  std::vector<uint32_t> osh(ord.size());
  std::vector<double> otr(12 * ord.size());
  for (size_t k = 0; k < ord.size(); ++k) {
    osh[k] = ctx->obs_shape[ord[k]];
    std::copy(&ctx->obs_tr[12 * ord[k]], &ctx->obs_tr[12 * ord[k]] + 12, &otr[12 * k]);
  }
  // linked cells per sim (Grains.cpp:226-247, LinkedCell.cpp:16-29)
  ctx->grids.assign(ns, SimGrid());
  std::vector<double> lc(ns, 0.0), rmean(ns, 0.0);  // largest radius, sum of the radii
  std::vector<uint64_t> rnum(ns, 0);
  for (uint64_t i = 0; i < ctx->n; ++i) {
    const HostShape& h = ctx->shapes[ctx->pshape[i]];
    const uint32_t s = ctx->psim[i];
    const double rc = quirks ? h.rc : h.rc_exact;
    lc[s] = std::max(lc[s], rc);
    rmean[s] += rc;
    ++rnum[s];
  }
  uint64_t base = 0;
  const uint32_t per = ctx->nmat * (ctx->nmat + 1) / 2;
  for (uint32_t s = 0; s < ns; ++s) {
    const grains_sim_t& S = ctx->sims[s];
    SimGrid& g = ctx->grids[s];
    double h = S.cell_size;
    if (!(h > 0)) h = std::max(1.0, S.cell_size_factor) * 2.0 * lc[s];
    if (!(h > 0)) return fail(ctx, GRAINS_EINVAL, "sim " + std::to_string(s) + ": zero cell size");
    g.h = h;
    for (int k = 0; k < 3; ++k) {
      g.lo[k] = S.domain_min[k];
      g.hi[k] = S.domain_max[k];
      g.L[k] = S.domain_max[k] - S.domain_min[k];
      g.g[k] = S.gravity[k];
      double c = kEps;
      c += S.domain_max[k] - S.domain_min[k];
      c /= h;
      if (!(c >= 1.0) || c > 4e9) return fail(ctx, GRAINS_EINVAL, "sim " + std::to_string(s) + ": bad domain");
      g.n3[k] = (uint32_t)c;
      if (((S.periodic >> k) & 1) && g.n3[k] < 3)
        return fail(ctx, GRAINS_EINVAL, "periodic direction needs >= 3 cells");
    }
    g.periodic = S.periodic;
    if (S.contact_table < 0 || (uint32_t)S.contact_table >= ctx->ntables)
      return fail(ctx, GRAINS_EINVAL, "contact table index out of range");
    g.table = (uint32_t)S.contact_table * per;
    g.base = (uint32_t)base;
    base += (uint64_t)g.n3[0] * g.n3[1] * g.n3[2];
    if (base >= (1ull << 32) - 1) return fail(ctx, GRAINS_EINVAL, "too many cells");
    g.obs_begin = g.obs_end = 0;
  }
  for (size_t k = 0; k < ord.size(); ++k) {
    SimGrid& g = ctx->grids[ctx->obs_sim[ord[k]]];
    if (g.obs_end == g.obs_begin) g.obs_begin = (uint32_t)k;
    g.obs_end = (uint32_t)k + 1;
  }
  // The search's cells: the reference's, or wider where the lists' reach --
  // the largest two radii and the skin -- asks for it.  The skin is a tenth of
  // the sim's mean radius: on the superquadric beds it grows the lists by a
  // fifth, and grains at 0.2 m/s (dt = 1e-6) take about 60 steps to use it up.
  // Measured (ms/step, skin 0.02 / 0.05 / 0.1 / 0.2 of the mean radius): bed of
  // 10^6 at rest 0.355 / 0.364 / 0.380 / 0.400, 50,653 agitated grains 0.456 /
  // 0.452 / 0.447 / 0.447, 100,003 polyhedra 0.290 / 0.279 / 0.270 / 0.273, 64
  // beds (369,564) 0.358 / 0.356 / 0.354 / 0.367; lists built every step:
  // 0.58, 0.52, 0.40, 0.58.
  // A periodic axis that would hold fewer than three such cells leaves the
  // whole context without a skin (set_search).
  bool skin_fits = true;
  uint64_t sbase = 0;
  ctx->sgrids = ctx->grids;
  for (uint32_t s = 0; s < ns; ++s) {
    SimGrid& g = ctx->sgrids[s];
    const double skin = rnum[s] ? 0.1 * rmean[s] / (double)rnum[s] : 0.0;
    const double h = std::max(g.h, (2.0 * lc[s] + skin) * (1.0 + 1e-9));
    for (int k = 0; k < 3; ++k)
      if ((rnum[s] && !(skin > 1e-9 * g.L[k])) || (((g.periodic >> k) & 1) && g.L[k] < 3.0 * h)) skin_fits = false;
    if (h != g.h)
      for (int k = 0; k < 3; ++k) g.n3[k] = (uint32_t)std::max(1.0, g.L[k] / h);
    g.h = h;
    g.half_skin = 0.5 * skin;
    g.move2 = 0.25 * skin * skin * (1.0 - 1e-6) * (1.0 - 1e-6);
    g.base = (uint32_t)sbase;
    sbase += (uint64_t)g.n3[0] * g.n3[1] * g.n3[2];
    ctx->grids[s].move2 = g.move2;
  }
  {
    int ref = 1;
    while (ref < 32 && (1ull << ref) < base) ++ref;
    ctx->ref_passes = (ref + kRadixMaxBits - 1) / kRadixMaxBits;
    ctx->ref_digit_bits = std::max(8, (ref + ctx->ref_passes - 1) / ctx->ref_passes);
  }
  // shape tables
  const size_t S = ctx->shapes.size();
  std::vector<ShapeNP<double>> np64(S);
  std::vector<ShapeNP<float>> np32(S);
  std::vector<ShapeDyn> dyn(S);
  std::vector<double> rcpf(S), v64, cv64;
  for (size_t i = 0; i < S; ++i) {
    const HostShape& h = ctx->shapes[i];
    int32_t voff = (int32_t)(v64.size() / 3);
    np64[i] = to_np<double>(h, quirks, voff);
    np32[i] = to_np<float>(h, quirks, voff);
    ShapeDyn& y = dyn[i];
    y = ShapeDyn{};
    y.mass = h.mass;
    for (int k = 0; k < 3; ++k) {
      constexpr int on[3] = {0, 3, 5}, off[3] = {1, 2, 4};
      y.diag[k] = h.inertia[on[k]], y.inv_diag[k] = h.inv[on[k]];
      y.off[k] = h.inertia[off[k]], y.inv_off[k] = h.inv[off[k]];
      if (y.off[k] != 0.0 || y.inv_off[k] != 0.0) y.off_axis = 1.0;
    }
    rcpf[i] = quirks ? h.rc : h.rc_exact;
    v64.insert(v64.end(), h.verts.begin(), h.verts.end());
    cv64.insert(cv64.end(), h.core_verts.begin(), h.core_verts.end());
  }
  if (v64.empty()) v64.assign(3, 0.0), cv64.assign(3, 0.0);
  std::vector<float> v32(v64.begin(), v64.end()), cv32(cv64.begin(), cv64.end());
  std::vector<HookeP<double>> hk64(ctx->tables.size());
  std::vector<HookeP<float>> hk32(ctx->tables.size());
  for (size_t i = 0; i < ctx->tables.size(); ++i) {
    const grains_hooke_t& t = ctx->tables[i];
    double muen = std::log(t.en) / std::sqrt(kPi * kPi + std::log(t.en) * std::log(t.en));
    hk64[i] = {t.kn, t.en, t.etat, t.muc, t.kr, muen};
    hk32[i] = {(float)t.kn, (float)t.en, (float)t.etat, (float)t.muc, (float)t.kr, (float)muen};
  }
  auto& L = ctx->allocs;
  const uint64_t n = ctx->n;  // (the arrays by cell hold the search's cells with and without a skin: never more than base)
  const uint32_t K = (uint32_t)ctx->cfg.max_neighbors;
  const uint64_t ecap = n * K;
  const uint64_t ntiles = (n + kTile - 1) / kTile;
  // the narrow phase's launch may hold up to 64 blocks per CU of up to 256
  // threads (grains_set_launch); the screen's queue has one segment per block
  const uint64_t max_nb = (uint64_t)cu_count() * kMaxNarrowPerCu;
  const uint64_t nhist = (uint64_t)kRadixMaxDigits * ntiles;  // histogram of the widest digit
  const uint64_t nblk = std::max(std::max((n + kTile - 1) / kTile, (nhist + kTile - 1) / kTile),
                                 std::max((max_nb + kTile) / kTile, (base + kTile) / kTile)) +
                        2;
  // entry results in FP64 for the plain path and for FP32-mixed with FP64
  // contact geometry (whose contacts all come from FP64 re-runs)
  const bool res64 = ctx->cfg.precision == GRAINS_FP64 || (ctx->cfg.flags & GRAINS_FP64_CONTACTS);
  const size_t res_sz = res64 ? sizeof(PairRes<double>) : sizeof(PairRes<float>);
  int rc;
  ShapeNP<double>* p64;
  ShapeNP<float>* p32;
  SqPow* psq;
  ShapeDyn* pdyn;
  double *prc, *pv64, *pcv64, *potr;
  float *pv32, *pcv32;
  HookeP<double>* ph64;
  HookeP<float>* ph32;
  SimGrid *pgr, *psg;
  uint32_t* posh;
  if ((rc = dalloc(ctx, &p64, S * sizeof(ShapeNP<double>), L)) || (rc = dalloc(ctx, &p32, S * sizeof(ShapeNP<float>), L)) ||
      (rc = dalloc(ctx, &psq, S * sizeof(SqPow), L)) || (rc = dalloc(ctx, &pdyn, S * sizeof(ShapeDyn), L)) || (rc = dalloc(ctx, &prc, S * sizeof(double), L)) ||
      (rc = dalloc(ctx, &pv64, v64.size() * sizeof(double), L)) || (rc = dalloc(ctx, &pcv64, cv64.size() * sizeof(double), L)) ||
      (rc = dalloc(ctx, &pv32, v32.size() * sizeof(float), L)) || (rc = dalloc(ctx, &pcv32, cv32.size() * sizeof(float), L)) ||
      (rc = dalloc(ctx, &ph64, hk64.size() * sizeof(HookeP<double>), L)) ||
      (rc = dalloc(ctx, &ph32, hk32.size() * sizeof(HookeP<float>), L)) ||
      (rc = dalloc(ctx, &pgr, ns * sizeof(SimGrid), L)) || (rc = dalloc(ctx, &psg, ns * sizeof(SimGrid), L)) ||
      (rc = dalloc(ctx, &d.skey, n * 4, L)) || (rc = dalloc(ctx, &d.rkey, n * 4, L)) || (rc = dalloc(ctx, &d.rcs, n * 8, L)) || (rc = dalloc(ctx, &posh, (osh.size() + 1) * sizeof(uint32_t), L)) ||
      (rc = dalloc(ctx, &potr, (otr.size() + 12) * sizeof(double), L)) ||
      (rc = dalloc(ctx, &d.key, n * 4, L)) || (rc = dalloc(ctx, &d.keyA, n * 4, L)) || (rc = dalloc(ctx, &d.idxA, n * 4, L)) ||
      (rc = dalloc(ctx, &d.keyB, n * 4, L)) || (rc = dalloc(ctx, &d.idxB, n * 4, L)) || (rc = dalloc(ctx, &d.rank, n * 4, L)) ||
      (rc = dalloc(ctx, &d.cell_off, (base + 1) * 4, L)) ||
      (rc = dalloc(ctx, &d.bp, n * sizeof(double4), L)) || (rc = dalloc(ctx, &d.pk, n * sizeof(PoseRec), L)) ||
      (rc = dalloc(ctx, &d.vk, n * sizeof(VelRec), L)) || (rc = dalloc(ctx, &d.rws, n * 8, L)) ||
      (rc = dalloc(ctx, &d.bp32, n * sizeof(float4), L)) ||
      (rc = dalloc(ctx, &d.cell_sph, (base + 1) * sizeof(float4), L)) ||
      (rc = dalloc(ctx, &d.half_goff, (base + 1) * 4, L)) || (rc = dalloc(ctx, &d.half_glist, n * 4, L)) ||
      (rc = dalloc(ctx, &d.hist, (nhist + 1) * 4, L)) || (rc = dalloc(ctx, &d.scan_blocks, nblk * 4, L)) ||
      (rc = dalloc(ctx, &d.cand, ecap * 4, L)) || (rc = dalloc(ctx, &d.cand_count, n * 4, L)) ||
      (rc = dalloc(ctx, &d.entry_off, (n + 1) * 4, L)) || (rc = dalloc(ctx, &d.pair_i, ecap * 4, L)) ||
      (rc = dalloc(ctx, &d.pair_j, ecap * 4, L)) || (rc = dalloc(ctx, &d.pair_flag, ecap * 4, L)) ||
      (rc = dalloc(ctx, &d.pair_res, ecap * res_sz, L)) || (rc = dalloc(ctx, &d.refine_list, ecap * 4, L)) ||
      (rc = dalloc(ctx, &d.refine_count, 16, L)) || (rc = dalloc(ctx, &d.obs_list, (n + 1) * 4, L)) ||
      (rc = dalloc(ctx, &d.obs_list2, n * 4, L)) ||
      (rc = dalloc(ctx, &d.obs_count, 16, L)) || (rc = dalloc(ctx, &d.pend, n * 4, L)) ||
      (rc = dalloc(ctx, &d.pend_list, n * 4, L)) || (rc = dalloc(ctx, &d.sort_state, 16, L)) ||
      (rc = dalloc(ctx, &d.mv_list, kMaxMovers * 4, L)) || (rc = dalloc(ctx, &d.mv_keys, kMaxMovers * 8, L)) ||
      (rc = dalloc(ctx, &d.mv_old, kMaxMovers * 4, L)) || (rc = dalloc(ctx, &d.mv_dst, kMaxMovers * 4, L)) ||
      (rc = dalloc(ctx, &d.defer_list, defer_words(ecap) * 4, L)) ||
      (rc = dalloc(ctx, &d.defer_count, kDeferQueues * 64, L)) || (rc = dalloc(ctx, &d.counters, kWordBytes, L)))
    return rc;
  d.gjk_rec = nullptr;
  if ((rc = dalloc(ctx, &d.log, sizeof(StateLog), L))) return rc;
  launch_fill_u32((uint32_t*)d.log, sizeof(StateLog) / 4, 0u, ctx->stream);
  d.hk = nullptr;
  if (d.ab_hist && (rc = dalloc(ctx, &d.hk, 12 * n * sizeof(double), L))) return rc;
  d.pend_count = d.obs_count + 1;
  d.obs_count2 = d.obs_count + 2;
  d.queue_next = d.obs_count + 3;
  d.nl = (uint32_t*)((unsigned char*)d.counters + kCounterBytes);
  // warm-start records: two buffers of ecap = K x N, zeroed (no direction)
  d.warm = ((ctx->cfg.flags & GRAINS_WARM_START) && ctx->cfg.precision == GRAINS_FP32_MIXED &&
            !(ctx->cfg.flags & GRAINS_REF_QUIRKS))
               ? 1
               : 0;
  d.ws = nullptr;
  d.ws_nb = nullptr;
  d.ws_par = nullptr;
  if (d.warm) {
    if ((rc = dalloc(ctx, &d.ws, 2 * ecap * sizeof(float4), L)) || (rc = dalloc(ctx, &d.ws_nb, 2 * n * sizeof(uint2), L)) ||
        (rc = dalloc(ctx, &d.ws_par, 16, L)))
      return rc;
    launch_fill_u32((uint32_t*)d.ws, 2 * ecap * 4, 0u, ctx->stream);
    launch_fill_u32((uint32_t*)d.ws_nb, 4 * n, 0u, ctx->stream);
    launch_fill_u32(d.ws_par, 4, 0u, ctx->stream);
  }
  GR_HIP(hipMemcpy(p64, np64.data(), S * sizeof(ShapeNP<double>), hipMemcpyHostToDevice));
  GR_HIP(hipMemcpy(p32, np32.data(), S * sizeof(ShapeNP<float>), hipMemcpyHostToDevice));
  launch_sq_pow(p64, psq, S, ctx->stream);
  GR_HIP(hipMemcpy(pdyn, dyn.data(), S * sizeof(ShapeDyn), hipMemcpyHostToDevice));
  GR_HIP(hipMemcpy(prc, rcpf.data(), S * sizeof(double), hipMemcpyHostToDevice));
  GR_HIP(hipMemcpy(pv64, v64.data(), v64.size() * sizeof(double), hipMemcpyHostToDevice));
  GR_HIP(hipMemcpy(pcv64, cv64.data(), cv64.size() * sizeof(double), hipMemcpyHostToDevice));
  GR_HIP(hipMemcpy(pv32, v32.data(), v32.size() * sizeof(float), hipMemcpyHostToDevice));
  GR_HIP(hipMemcpy(pcv32, cv32.data(), cv32.size() * sizeof(float), hipMemcpyHostToDevice));
  GR_HIP(hipMemcpy(ph64, hk64.data(), hk64.size() * sizeof(HookeP<double>), hipMemcpyHostToDevice));
  GR_HIP(hipMemcpy(ph32, hk32.data(), hk32.size() * sizeof(HookeP<float>), hipMemcpyHostToDevice));
  GR_HIP(hipMemcpy(pgr, ctx->grids.data(), ns * sizeof(SimGrid), hipMemcpyHostToDevice));
  set_search(ctx, skin_fits);
  GR_HIP(hipMemcpy(psg, search_grids(ctx).data(), ns * sizeof(SimGrid), hipMemcpyHostToDevice));
  if (!osh.empty()) {
    GR_HIP(hipMemcpy(posh, osh.data(), osh.size() * sizeof(uint32_t), hipMemcpyHostToDevice));
    GR_HIP(hipMemcpy(potr, otr.data(), otr.size() * sizeof(double), hipMemcpyHostToDevice));
  }
  d.np64 = p64;
  d.np32 = p32;
  d.sq64 = psq;
  d.dyn = pdyn;
  d.rc_pf = prc;
  d.verts64 = pv64;
  d.cverts64 = pcv64;
  d.verts32 = pv32;
  d.cverts32 = pcv32;
  d.hooke64 = ph64;
  d.hooke32 = ph32;
  d.grids = pgr;
  d.sgrids = psg;
  d.keep_torce = 0;
  d.obs_shape = posh;
  d.obs_tr = potr;
  d.nsims = ns;
  d.nobs = (uint32_t)osh.size();
  d.nmat = ctx->nmat;
  d.K = K;
  d.ecap = ecap;
  d.dt = ctx->cfg.dt;
  d.flags = ctx->cfg.flags;
  d.gjk_rel = ctx->cfg.gjk_rel_tol;
  d.gjk_rel64 = ctx->cfg.gjk_rel_tol_fp64;
  d.res64 = ctx->cfg.precision == GRAINS_FP32_MIXED && (ctx->cfg.flags & GRAINS_FP64_CONTACTS) ? 1 : 0;
  d.precision = ctx->cfg.precision;
  d.integrator = ctx->cfg.integrator;
  d.block = (uint32_t)ctx->cfg.block_size;
  d.narrow_blocks = (uint32_t)(cu_count() * ctx->cfg.narrow_blocks_per_cu);
  d.split = ctx->cfg.narrow_passes == 2 ? 1 : 0;
  // a small bed sorts in one block (measured: 1,000 particles 0.113 ->
  // 0.094 ms/step; 2,048, 4,096 and 8,192 slower than the radix passes and
  // the merge: 0.267, 0.352, 0.425 against 0.255, 0.320, 0.338 ms);
  // GRAINS_SMALL_SORT_MAX sets the largest such bed, up to kSmallSort (0:
  // always the radix passes and the merge)
  uint64_t small_max = kSmallSortDefault;
  if (const char* e = std::getenv("GRAINS_SMALL_SORT_MAX")) small_max = std::strtoull(e, nullptr, 10);
  d.small_sort = n <= std::min<uint64_t>(small_max, kSmallSort) ? 1 : 0;
  launch_fill_u32(d.cand_count, n, 0u, ctx->stream);
  launch_fill_u32(d.entry_off, n + 1, 0u, ctx->stream);
  launch_fill_u32(d.refine_count, 4, 0u, ctx->stream);
  launch_fill_u32(d.sort_state, 4, 0u, ctx->stream);
  launch_fill_u32(d.obs_count, 4, 0u, ctx->stream);
  launch_fill_u32(d.defer_count, kDeferQueues * 16, 0u, ctx->stream);
  set_defer_cap(ctx);
  launch_fill_u32((uint32_t*)d.counters, kWordBytes / 4, 0u, ctx->stream);
  GR_HIP(hipGetLastError());
  GR_HIP(hipStreamSynchronize(ctx->stream));
  ctx->layout_ok = true;
  ctx->keys_s = ctx->idx_s = nullptr;  // no lists yet
  ctx->lists_ok = false;
  ctx->skin_back = false;
  ctx->interval = 8;
  ctx->interval_known = false;
  return GRAINS_OK;
}

extern "C" int grains_set_state(grains_ctx_t* ctx, const double* pos, const double* quat, const double* vel,
                                const double* omega, uint64_t n) {
  if (!ctx) return GRAINS_EINVAL;
  if (n != ctx->n || !n) return fail(ctx, GRAINS_EINVAL, "particle count mismatch");
  std::vector<double> buf(4 * n);
  auto put = [&](const double* src, double* dst, int comps) -> int {
    if (!src) return GRAINS_OK;
    for (uint64_t i = 0; i < n; ++i)
      for (int k = 0; k < comps; ++k) buf[k * n + i] = src[comps * i + k];
    GR_HIP(hipMemcpy(dst, buf.data(), comps * n * sizeof(double), hipMemcpyHostToDevice));
    return GRAINS_OK;
  };
  int rc;
  if ((rc = put(pos, ctx->d.pos, 3)) || (rc = put(quat, ctx->d.quat, 4)) || (rc = put(vel, ctx->d.vel, 3)) ||
      (rc = put(omega, ctx->d.omega, 3)) || (rc = warm_reset(ctx)))
    return rc;
  return hist_reset(ctx);
}

constexpr uint64_t kRowsMax = 1u << 18;        // particles per pinned buffer (27 MB)
constexpr uint64_t kRowsPerThread = 1u << 14;  // particles worth a thread of their own (1.7 MB)

// a part of a get_state: particles [i0, i0 + m) from the rows in `rows`
struct StateDst {
  double *pos, *quat, *vel, *omega;
};
static void copy_rows(const StateDst& o, const double* rows, uint64_t i0, uint64_t m, uint64_t a, uint64_t b) {
  auto put = [&](double* dst, uint64_t base, uint64_t comps) {
    if (dst) std::memcpy(dst + comps * (i0 + a), rows + base * m + comps * a, comps * (b - a) * sizeof(double));
  };
  put(o.pos, 0, 3), put(o.quat, 3, 4), put(o.vel, 7, 3), put(o.omega, 10, 3);
}
// f(a, b) for the parts [a, b) of [0, n), at least `per` long, by up to
// eight threads.
template <class F>
static void in_parts(uint64_t n, uint64_t per, const F& f) {
  const uint64_t parts =
      std::min<uint64_t>(std::max(1u, std::min(8u, std::thread::hardware_concurrency())), n / per + 1);
  uint64_t left = parts;  // parts [0, left) are this thread's
  std::vector<std::thread> th;
  try {
    th.reserve(parts);
    while (left > 1) {
      const uint64_t a = n * (left - 1) / parts, b = n * left / parts;
      th.emplace_back([=, &f] { f(a, b); });
      --left;
    }
  } catch (const std::exception&) {  // no more threads: the rest is done here
  }
  f(0, n * left / parts);
  for (std::thread& t : th) t.join();
}
// The same by several threads: a caller's array that has not been written
// before costs a page fault per 4 KB, 104 MB of them 20 ms on one thread.
static void copy_rows_threads(const StateDst& o, const double* rows, uint64_t i0, uint64_t m) {
  in_parts(m, kRowsPerThread, [&](uint64_t a, uint64_t b) { copy_rows(o, rows, i0, m, a, b); });
}

static void free_rows(grains_ctx* ctx) {
  for (int k = 0; k < 2; ++k) {
    if (ctx->rows[k]) (void)hipHostFree(ctx->rows[k]);
    ctx->rows[k] = nullptr;
  }
  ctx->rows_cap = 0;
}
static bool alloc_rows(grains_ctx* ctx, uint64_t cap, int count) {
  for (int k = 0; k < count; ++k)
    if (hipHostMalloc((void**)&ctx->rows[k], 13 * cap * sizeof(double), hipHostMallocDefault) != hipSuccess) {
      (void)hipGetLastError();
      free_rows(ctx);
      return false;
    }
  ctx->rows_cap = cap;
  return true;
}

// The planes turn into rows on the device, written into one of two pinned
// buffers while the other is copied out: 10^6 particles 20 -> 3.7 ms (planes
// copied to pageable memory and turned into rows by the host).
extern "C" int grains_get_state(grains_ctx_t* ctx, double* pos, double* quat, double* vel, double* omega,
                                uint64_t n) {
  if (!ctx) return GRAINS_EINVAL;
  if (n != ctx->n || !n) return fail(ctx, GRAINS_EINVAL, "particle count mismatch");
  const StateDst out = {pos, quat, vel, omega};
  std::lock_guard<std::mutex> lock(ctx->rows_mu);
  if (ctx->rows_cap < std::min(n, kRowsMax) || (n > ctx->rows_cap && !ctx->rows[1])) {
    free_rows(ctx);
    uint64_t cap = std::min(n, kRowsMax);
    // less at a time where so much cannot be pinned
    while (!alloc_rows(ctx, cap, cap < n ? 2 : 1)) {
      if (cap <= 256) return fail(ctx, GRAINS_EDEVICE, "no pinned memory for the state");
      cap = std::max<uint64_t>(256, cap / 2);
    }
  }
  const uint64_t cap = ctx->rows_cap;
  hipStream_t s = ctx->stream;
  auto start = [&](uint64_t c) -> hipError_t {
    launch_state_rows(ctx->d, c * cap, std::min(cap, n - c * cap), ctx->rows[c & 1], s);
    hipError_t e = hipGetLastError();
    return e != hipSuccess ? e : hipEventRecord(ctx->rows_ev[c & 1], s);
  };
  const uint64_t chunks = (n + cap - 1) / cap;
  GR_HIP(start(0));
  for (uint64_t c = 0; c < chunks; ++c) {
    GR_HIP(hipEventSynchronize(ctx->rows_ev[c & 1]));
    if (c + 1 < chunks) GR_HIP(start(c + 1));
    copy_rows_threads(out, ctx->rows[c & 1], c * cap, std::min(cap, n - c * cap));
  }
  return GRAINS_OK;
}

// Transform3 buffers <-> (origin, quaternion).  The quaternion of a basis is
// taken with the four-branch rule of Quaternion::setQuaternion(Matrix3)
// (Quaternion.cpp:125-169).
extern "C" int grains_set_transforms(grains_ctx_t* ctx, const double* t, uint64_t n) {
  if (!ctx || !t) return GRAINS_EINVAL;
  if (n != ctx->n) return fail(ctx, GRAINS_EINVAL, "particle count mismatch");
  std::vector<double> pos(3 * n), q(4 * n);
  for (uint64_t i = 0; i < n; ++i) {
    const double* b = t + 12 * i;
    enum { XX, XY, XZ, YX, YY, YZ, ZX, ZY, ZZ };
    double qx = 0, qy = 0, qz = 0, qw = 1, den;
    if (b[YY] > -b[ZZ] && b[XX] > -b[YY] && b[XX] > -b[ZZ]) {
      den = std::pow(1.0 + b[XX] + b[YY] + b[ZZ], 0.5);
      qw = 0.5 * den;
      qx = 0.5 * (b[ZY] - b[YZ]) / den;
      qy = 0.5 * (b[XZ] - b[ZX]) / den;
      qz = 0.5 * (b[YX] - b[XY]) / den;
    } else if (b[YY] < -b[ZZ] && b[XX] > b[YY] && b[XX] > b[ZZ]) {
      den = std::pow(1.0 + b[XX] - b[YY] - b[ZZ], 0.5);
      qw = 0.5 * (b[ZY] - b[YZ]) / den;
      qx = 0.5 * den;
      qy = 0.5 * (b[XY] + b[YX]) / den;
      qz = 0.5 * (b[ZX] + b[XZ]) / den;
    } else if (b[YY] > b[ZZ] && b[XX] < b[YY] && b[XX] < -b[ZZ]) {
      den = std::pow(1.0 - b[XX] + b[YY] - b[ZZ], 0.5);
      qw = 0.5 * (b[XZ] - b[ZX]) / den;
      qx = 0.5 * (b[XY] + b[YX]) / den;
      qy = 0.5 * den;
      qz = 0.5 * (b[YZ] + b[ZY]) / den;
    } else if (b[YY] < b[ZZ] && b[XX] < -b[YY] && b[XX] < b[ZZ]) {
      den = std::pow(1.0 - b[XX] - b[YY] + b[ZZ], 0.5);
      qw = 0.5 * (b[YX] - b[XY]) / den;
      qx = 0.5 * (b[ZX] + b[XZ]) / den;
      qy = 0.5 * (b[YZ] + b[ZY]) / den;
      qz = 0.5 * den;
    }
    q[4 * i] = qx, q[4 * i + 1] = qy, q[4 * i + 2] = qz, q[4 * i + 3] = qw;
    pos[3 * i] = b[9], pos[3 * i + 1] = b[10], pos[3 * i + 2] = b[11];
  }
  return grains_set_state(ctx, pos.data(), q.data(), nullptr, nullptr, n);
}

extern "C" int grains_get_transforms(grains_ctx_t* ctx, double* t, uint64_t n) {
  if (!ctx || !t) return GRAINS_EINVAL;
  std::vector<double> pos(3 * n), q(4 * n);
  int rc = grains_get_state(ctx, pos.data(), q.data(), nullptr, nullptr, n);
  if (rc) return rc;
  for (uint64_t i = 0; i < n; ++i) {
    M3<double> R = rot(Qt<double>{q[4 * i], q[4 * i + 1], q[4 * i + 2], q[4 * i + 3]});
    std::copy(R.m, R.m + 9, t + 12 * i);
    t[12 * i + 9] = pos[3 * i], t[12 * i + 10] = pos[3 * i + 1], t[12 * i + 11] = pos[3 * i + 2];
  }
  return GRAINS_OK;
}

// phase marker: an event on the stream when profiling (never while capturing)
static void mark(grains_ctx* ctx) {
  if (!ctx->profiling || ctx->capturing) return;
  if (ctx->pev_used == ctx->pev.size()) {
    hipEvent_t e;
    if (hipEventCreate(&e) != hipSuccess) {
      ctx->profiling = false;
      return;
    }
    ctx->pev.push_back(e);
  }
  (void)hipEventRecord(ctx->pev[ctx->pev_used++], ctx->stream);
}

// the neighbour lists built from the current positions, enqueued on
// ctx->stream (also what a graph captures)
static void enqueue_build(grains_ctx* ctx) {
  DevScene& d = ctx->d;
  hipStream_t s = ctx->stream;
  // (the sort's output pair: the last of its ping-pong passes; the previous
  // order's keys: where the last sort left them)
  launch_hash(d, (d.small_sort || (ctx->passes & 1)) ? d.keyA : d.keyB, s);
  mark(ctx);
  launch_sort(d, ctx->passes, ctx->digit_bits, &ctx->keys_s, &ctx->idx_s, s);
  mark(ctx);
  d.sidx = ctx->idx_s;
  launch_cells(d, ctx->keys_s, ctx->idx_s, s);
  mark(ctx);
  launch_candidates(d, ctx->keys_s, s);
  mark(ctx);
  launch_scan(d.cand_count, d.entry_off, d.n, d.scan_blocks, s, d.K);
  launch_expand(d, s);
  mark(ctx);
}

// one step over the lists (returning at once, kernel by kernel, when they no
// longer hold), after a build when `build`
static void enqueue_step(grains_ctx* ctx, bool build) {
  DevScene& d = ctx->d;
  hipStream_t s = ctx->stream;
  mark(ctx);
  if (build)
    enqueue_build(ctx);
  else
    for (int k = 0; k < 5; ++k) mark(ctx);  // the build's phases: nothing
  // the integration split around the narrow phase's second pass: two
  // passes (physics semantics), the step not profiled phase by phase; a
  // small bed's integration is too short to be worth the second stream, and
  // spheres in FP64 have no second pass
  const bool split = d.n > kWideIntegrate && !(d.balls && d.precision == GRAINS_FP64) && d.split > 0 && !(d.flags & GRAINS_REF_QUIRKS) && !ctx->adj_rec &&
                     !(ctx->profiling && !ctx->capturing);
  if (d.precision == GRAINS_FP64 && split) {
    launch_narrow64(d, 0, s);
    (void)hipEventRecord(ctx->ev_fork, s);
    (void)hipStreamWaitEvent(ctx->side, ctx->ev_fork, 0);
    launch_integrate64(d, ctx->side, 1);
    (void)hipEventRecord(ctx->ev_join, ctx->side);
    launch_narrow64(d, 1, s);
    (void)hipStreamWaitEvent(s, ctx->ev_join, 0);
    launch_integrate64(d, s, 2);
  } else if (d.precision == GRAINS_FP64) {
    launch_narrow64(d, 0, s);
    mark(ctx);
    launch_narrow64(d, 1, s);
    mark(ctx);
    mark(ctx);
    launch_integrate64(d, s);
  } else if (split) {
    // the particles the screen settled are integrated on the side stream
    // while the complete pass and the FP64 re-runs settle the others
    launch_narrow32(d, 0, s);
    (void)hipEventRecord(ctx->ev_fork, s);
    launch_narrow32(d, 1, s);  // first: its few long searches must not wait for room beside the integration
    (void)hipStreamWaitEvent(ctx->side, ctx->ev_fork, 0);
    launch_integrate32(d, ctx->side, 1);
    (void)hipEventRecord(ctx->ev_join, ctx->side);
    launch_refine64(d, s);
    (void)hipStreamWaitEvent(s, ctx->ev_join, 0);
    launch_integrate32(d, s, 2);
  } else {
    launch_narrow32(d, 0, s);
    mark(ctx);
    launch_narrow32(d, 1, s);
    mark(ctx);
    launch_refine64(d, s);
    mark(ctx);
    launch_integrate32(d, s);
  }
  if (ctx->adj_rec && !d.keep_torce) launch_log_state(d, s);
  mark(ctx);
}

// the counters and list words, read back (the stream is then idle)
static int read_words(grains_ctx* ctx, uint32_t* nl) {
  GR_HIP(hipMemcpyAsync(ctx->host_words, ctx->d.counters, kWordBytes, hipMemcpyDeviceToHost, ctx->stream));
  GR_HIP(hipStreamSynchronize(ctx->stream));
  std::memcpy(nl, ctx->host_words + kCounterBytes, kNlWords * 4);
  return GRAINS_OK;
}

static void read_stats(grains_ctx* ctx, uint32_t steps) {
  const unsigned long long* slots = (const unsigned long long*)ctx->host_words;
  unsigned long long c[kNumCounters];
  for (int k = 0; k < kNumCounters; ++k) {
    c[k] = 0;
    for (int j = 0; j < kCntSlots; ++j) {
      const unsigned long long v = slots[(size_t)k * kCntSlots + j];
      c[k] = (k == kCntMaxCand || k == kCntMaxIters || k == kCntRefMaxIters) ? std::max(c[k], v) : c[k] + v;
    }
  }
  grains_stats_t& st = ctx->stats;
  st.steps = steps;
  st.candidate_pairs = c[kCntCandidates];
  st.gjk_calls = c[kCntGjk];
  st.gjk_iterations = c[kCntGjkIters];
  st.contacts = c[kCntContacts];
  st.wall_contacts = c[kCntWall];
  st.out_of_domain = c[kCntOod];
  st.deep_contacts = c[kCntDeep];
  st.fp64_refines = c[kCntRefine];
  st.narrow_deferred = c[kCntDeferred];
  st.gjk_max_iterations = c[kCntMaxIters];
  st.fp64_near_refines = c[kCntNear];
  st.nonfinite_states = c[kCntNan];
  st.fp64_refine_iterations = c[kCntRefIters];
  st.fp64_refine_max_iterations = c[kCntRefMaxIters];
  st.neighbor_overflow = c[kCntOverflow];
  st.max_candidates = (uint32_t)c[kCntMaxCand];
  st.sort_passes = (uint32_t)ctx->ref_passes;
}

// The lists with their skin (on) or without, from the next build on.
static int use_skin(grains_ctx* ctx, bool on) {
  GR_HIP(hipStreamSynchronize(ctx->stream));
  set_search(ctx, on);
  const std::vector<SimGrid>& g = search_grids(ctx);
  GR_HIP(hipMemcpy((void*)ctx->d.sgrids, g.data(), g.size() * sizeof(SimGrid), hipMemcpyHostToDevice));
  launch_fill_u32(ctx->d.sort_state, 3, 0u, ctx->stream);  // the standing order is that of other cells
  ctx->lists_ok = false;
  drop_graph(ctx);  // captured kernels hold the flag
  return GRAINS_OK;
}

// ---- differentiation: recorded trajectory --------------------------------------
// the live state <-> 13 planes (pos 3, quat 4, vel 3, omega 3), on the stream
static int state_to(grains_ctx* ctx, double* dst) {
  GR_HIP(hipMemcpyAsync(dst, ctx->d.pos, 13 * ctx->n * 8, hipMemcpyDeviceToDevice, ctx->stream));
  return GRAINS_OK;
}
static int state_from(grains_ctx* ctx, const double* src) {
  GR_HIP(hipMemcpyAsync(ctx->d.pos, src, 13 * ctx->n * 8, hipMemcpyDeviceToDevice, ctx->stream));
  return GRAINS_OK;
}
// after recorded steps (never past a checkpoint): a checkpoint every
// adj_every steps, of the planes that its step has written (log_chunk)
static int adj_after_steps(grains_ctx* ctx, uint32_t steps) {
  ctx->adj_steps += steps;
  if (!steps || ctx->adj_steps % ctx->adj_every) return GRAINS_OK;
  double* cp;
  int rc = adj_dalloc(ctx, &cp, 13 * ctx->n * 8, ctx->adj_cp);
  if (rc) return rc;
  return state_to(ctx, cp);
}

// The states of a recorded trajectory's steps are kept beside its checkpoints
// while they fit kLogBytes (and the device), so that the sweep need not run
// them again: its block's memory (null: no more), and the place of the steps
// of a run of which `done` are taken.  The step that reaches the next
// checkpoint writes its results as a run's last does (target: the run's steps
// up to there): a checkpoint copies them, and a run that stops there because
// it finds no memory has them.
constexpr uint64_t kLogBytes = 4ull << 30;
static int log_chunk(grains_ctx* ctx, uint32_t done, uint32_t target) {
  const uint64_t K = ctx->adj_every, blk = ctx->adj_steps / K, bytes = 13 * ctx->n * 8 * K;
  while (ctx->adj_log.size() <= blk) {
    double* p = nullptr;
    const uint64_t used = ctx->adj_log_allocs.size() * bytes;
    if (!ctx->adj_log_off && K > 1 && bytes / K / 13 / 8 == ctx->n && bytes <= kLogBytes && used <= kLogBytes - bytes)
      (void)adj_spare(ctx, &p, bytes, ctx->adj_log_allocs);
    ctx->adj_log.push_back(p);
  }
  launch_log_set(ctx->d, {ctx->adj_log[blk], (int64_t)(ctx->adj_steps % K) - (int64_t)done, K}, target, ctx->stream);
  GR_HIP(hipGetLastError());
  return GRAINS_OK;
}

// Steps are launched in chunks of as many as the lists are expected to hold
// for; the kernels of a step whose lists no longer hold return at once, and
// after each chunk the host reads how many were taken, builds new lists when
// they ran out, and goes on.
static int take_steps(grains_ctx* ctx, uint32_t n_steps, bool graph) {
  int rc;
  hipStream_t s = ctx->stream;
  launch_run_begin(ctx->d, n_steps, !ctx->lists_ok, s);
  // 0: the lists' build; otherwise that many steps
  auto capture = [&](uint32_t steps, hipGraph_t* g, hipGraphExec_t* ge) -> int {
    if (*ge) return GRAINS_OK;
    ctx->capturing = true;
    GR_HIP(hipStreamBeginCapture(s, hipStreamCaptureModeThreadLocal));
    if (!steps) enqueue_build(ctx);
    for (uint32_t k = 0; k < steps; ++k) enqueue_step(ctx, false);
    hipError_t ec = hipStreamEndCapture(s, g);
    ctx->capturing = false;
    GR_HIP(ec);
    GR_HIP(hipGraphInstantiate(ge, *g, nullptr, nullptr, 0));
    return GRAINS_OK;
  };
  // profiled steps are launched one by one with their builds' phases
  auto build = [&]() -> int {
    if (!graph) {
      enqueue_build(ctx);
      return GRAINS_OK;
    }
    if (int r = capture(0, &ctx->graph_build, &ctx->graph_build_exec)) return r;
    GR_HIP(hipGraphLaunch(ctx->graph_build_exec, s));
    return GRAINS_OK;
  };
  auto steps = [&](uint32_t m) -> int {
    if (!graph) {
      for (uint32_t k = 0; k < m; ++k) enqueue_step(ctx, false);
      return GRAINS_OK;
    }
    const uint32_t chunk = ctx->graph_steps;
    if (chunk > 1 && m >= chunk) {
      if (int r = capture(chunk, &ctx->graph_multi, &ctx->graph_multi_exec)) return r;
      for (; m >= chunk; m -= chunk) GR_HIP(hipGraphLaunch(ctx->graph_multi_exec, s));
    }
    if (m)
      if (int r = capture(1, &ctx->graph, &ctx->graph_exec)) return r;
    for (; m; --m) GR_HIP(hipGraphLaunch(ctx->graph_exec, s));
    return GRAINS_OK;
  };
  ctx->pev_used = 0;
  GR_HIP(hipEventRecord(ctx->ev0, s));
  uint32_t done = 0, nl[kNlWords] = {0};
  while (done < n_steps) {
    uint32_t m = n_steps - done;
    if (ctx->adj_rec) {
      m = std::min<uint32_t>(m, ctx->adj_every - (uint32_t)(ctx->adj_steps % ctx->adj_every));
      if ((rc = log_chunk(ctx, done, done + m))) return rc;
    }
    const bool each = !ctx->d.skin || ctx->interval <= 1;  // lists for one step at a time
    if (each) {
      m = std::min(m, ctx->skin_back ? 1u : 64u);
      for (uint32_t k = 0; k < m; ++k) {
        if (ctx->profiling && !graph) {
          enqueue_step(ctx, true);
        } else {
          if ((rc = build()) || (rc = steps(1))) return rc;
        }
      }
      if (!ctx->skin_back) ctx->interval = 4;
    } else {
      bool fresh = !ctx->lists_ok;
      if (fresh) ctx->since_build = 0;
      m = std::min(m, ctx->interval > ctx->since_build ? ctx->interval - ctx->since_build : 1u);
      if (fresh && ctx->profiling && !graph) {
        enqueue_step(ctx, true);
        if ((rc = steps(m - 1))) return rc;
      } else if ((fresh && (rc = build())) || (rc = steps(m))) {
        return rc;
      }
    }
    GR_HIP(hipGetLastError());
    if (done + m == n_steps) GR_HIP(hipEventRecord(ctx->ev1, s));
    if ((rc = read_words(ctx, nl))) return rc;
    const uint32_t took = nl[kNlDone] - done;
    if (ctx->d.skin && nl[kNlOver]) {
      // a list outgrew max_neighbors with the skin, and the step's own
      // candidates may still fit; or centres lie outside a periodic side, and
      // the next step, which wraps them, takes the reference's cells
      if ((rc = use_skin(ctx, false))) return rc;
      ctx->skin_back = nl[kNlOver] == 3u;
    } else if (!took) {
      return fail(ctx, GRAINS_EDEVICE, "a step did not run");
    } else if (ctx->skin_back) {
      ctx->skin_back = false;
      if ((rc = use_skin(ctx, true))) return rc;
    } else {
      ctx->lists_ok = nl[kNlValid] != 0;
      ctx->since_build = each ? 1u : ctx->since_build + took;
      if (!each && !ctx->lists_ok) {
        ctx->interval = ctx->since_build;
        ctx->interval_known = true;
      } else if (!each && ctx->since_build >= ctx->interval) {
        // they outlast the estimate: a little more once a build has shown
        // how long they last, else twice as long
        ctx->interval = ctx->since_build + (ctx->interval_known ? 1 + ctx->since_build / 8 : ctx->since_build);
      }
    }
    done += took;
    if (ctx->adj_rec && (rc = adj_after_steps(ctx, took))) return rc;
  }
  if (!n_steps) {
    GR_HIP(hipEventRecord(ctx->ev1, s));
    if ((rc = read_words(ctx, nl))) return rc;
  }
  float ms = 0;
  GR_HIP(hipEventElapsedTime(&ms, ctx->ev0, ctx->ev1));
  for (int p = 0; p < GRAINS_NUM_PHASES; ++p) ctx->phase_ms[p] = 0;
  if (ctx->profiling && !graph) {
    const uint32_t per = GRAINS_NUM_PHASES + 1;
    for (uint32_t k = 0; k + per <= ctx->pev_used; k += per)
      for (int p = 0; p < GRAINS_NUM_PHASES; ++p) {
        float t = 0;
        GR_HIP(hipEventElapsedTime(&t, ctx->pev[k + p], ctx->pev[k + p + 1]));
        ctx->phase_ms[p] += t;
      }
  }
  read_stats(ctx, n_steps);
  ctx->stats.elapsed_ms = ms;
  if (ctx->stats.neighbor_overflow)
    return fail(ctx, GRAINS_EOVERFLOW, "candidate capacity max_neighbors exceeded (" +
                                           std::to_string(ctx->stats.max_candidates) + " needed)");
  return GRAINS_OK;
}

static int run_steps(grains_ctx* ctx, uint32_t n_steps, bool graph) {
  int rc = finalize(ctx);
  if (rc) return rc;
  rc = take_steps(ctx, n_steps, graph);
  if (rc) {
    // A run that stops early may have taken steps whose records are ahead of
    // the planes: these take them, and the next run starts from the planes.
    launch_store_state(ctx->d, ctx->stream);
    (void)hipStreamSynchronize(ctx->stream);
    ctx->lists_ok = false;
  }
  return rc;
}

extern "C" int grains_step(grains_ctx_t* ctx, uint32_t n_steps) {
  if (!ctx) return GRAINS_EINVAL;
  return run_steps(ctx, n_steps, false);
}

extern "C" int grains_step_graph(grains_ctx_t* ctx, uint32_t n_steps) {
  if (!ctx) return GRAINS_EINVAL;
  return run_steps(ctx, n_steps, true);
}

extern "C" int grains_set_graph_steps(grains_ctx_t* ctx, uint32_t steps) {
  if (!ctx) return GRAINS_EINVAL;
  if (steps < 1 || steps > 1000) return fail(ctx, GRAINS_EINVAL, "graph steps must be in [1, 1000]");
  if (steps != ctx->graph_steps) {
    ctx->graph_steps = steps;
    drop_graph(ctx);
  }
  return GRAINS_OK;
}

extern "C" int grains_set_launch(grains_ctx_t* ctx, int block_size, int narrow_blocks_per_cu) {
  if (!ctx) return GRAINS_EINVAL;
  if ((block_size != 64 && block_size != 128 && block_size != 256) || narrow_blocks_per_cu < 1 ||
      narrow_blocks_per_cu > kMaxNarrowPerCu)
    return fail(ctx, GRAINS_EINVAL, "block size must be 64, 128 or 256 and blocks per CU in [1, 64]");
  ctx->cfg.block_size = block_size;
  ctx->cfg.narrow_blocks_per_cu = narrow_blocks_per_cu;
  ctx->d.block = (uint32_t)block_size;
  ctx->d.narrow_blocks = (uint32_t)(cu_count() * narrow_blocks_per_cu);
  if (ctx->d.ecap) set_defer_cap(ctx);
  drop_graph(ctx);  // a captured step holds the old launch shape
  return GRAINS_OK;
}

extern "C" int grains_set_narrow_passes(grains_ctx_t* ctx, int passes) {
  if (!ctx || (passes != 1 && passes != 2)) return GRAINS_EINVAL;
  ctx->cfg.narrow_passes = passes;
  ctx->d.split = passes == 2 ? 1 : 0;
  drop_graph(ctx);  // a captured step holds the old pass structure
  return GRAINS_OK;
}

extern "C" int grains_set_candidate_staging(grains_ctx_t* ctx, int mode) {
  if (!ctx || mode < 0 || mode > 3) return GRAINS_EINVAL;
  ctx->cfg.candidate_staging = mode;
  if (ctx->layout_ok) set_search(ctx, ctx->d.skin != 0);
  drop_graph(ctx);  // a captured build holds the old kernel
  ctx->lists_ok = false;
  return GRAINS_OK;
}

extern "C" int grains_set_profiling(grains_ctx_t* ctx, int on) {
  if (!ctx) return GRAINS_EINVAL;
  ctx->profiling = on != 0;
  return GRAINS_OK;
}

extern "C" int grains_get_phase_times(grains_ctx_t* ctx, double* ms, int n) {
  if (!ctx || !ms || n < 0) return GRAINS_EINVAL;
  for (int p = 0; p < n && p < GRAINS_NUM_PHASES; ++p) ms[p] = ctx->phase_ms[p];
  return GRAINS_OK;
}

extern "C" int grains_get_cell_keys(grains_ctx_t* ctx, uint32_t* keys, uint32_t* sorted, uint64_t n) {
  if (!ctx) return GRAINS_EINVAL;
  if (n != ctx->n || !ctx->layout_ok || !ctx->idx_s) return fail(ctx, GRAINS_ESTATE, "no step run yet");
  GR_HIP(hipStreamSynchronize(ctx->stream));
  if (keys) GR_HIP(hipMemcpy(keys, ctx->d.key, n * 4, hipMemcpyDeviceToHost));
  if (sorted) {
    const uint32_t* order = launch_key_order(ctx->d, ctx->ref_passes, ctx->ref_digit_bits, ctx->stream);
    GR_HIP(hipGetLastError());
    GR_HIP(hipStreamSynchronize(ctx->stream));
    GR_HIP(hipMemcpy(sorted, order, n * 4, hipMemcpyDeviceToHost));
  }
  return GRAINS_OK;
}

extern "C" int grains_get_pairs(grains_ctx_t* ctx, int which, uint32_t* ij, uint64_t cap, uint64_t* m) {
  if (!ctx || !m) return GRAINS_EINVAL;
  if (!ctx->layout_ok || !ctx->idx_s) return fail(ctx, GRAINS_ESTATE, "no step run yet");
  GR_HIP(hipStreamSynchronize(ctx->stream));
  const uint64_t n = ctx->n;
  const uint32_t want = which == GRAINS_PAIRS_CONTACT ? kFlagContact : kFlagCand;
  const PairLists dev = launch_pair_lists(ctx->d, want, ij != nullptr, ctx->stream);
  GR_HIP(hipGetLastError());
  GR_HIP(hipStreamSynchronize(ctx->stream));
  uint32_t total = 0;
  GR_HIP(hipMemcpy(&total, dev.off + n, 4, hipMemcpyDeviceToHost));
  if (ij && total) {
    // (not vectors: their zeros cost as much as the copies into them)
    std::unique_ptr<uint32_t[]> off(new uint32_t[n + 1]), nb(new uint32_t[total]);
    GR_HIP(hipMemcpy(off.get(), dev.off, (n + 1) * 4, hipMemcpyDeviceToHost));
    GR_HIP(hipMemcpy(nb.get(), dev.nb, (uint64_t)total * 4, hipMemcpyDeviceToHost));
    in_parts(n, kRowsPerThread, [&](uint64_t a, uint64_t b) {
      for (uint64_t i = a; i < b; ++i)
        for (uint64_t k = off[i]; k < off[i + 1] && k < cap; ++k) ij[2 * k] = (uint32_t)i, ij[2 * k + 1] = nb[k];
    });
  }
  *m = total;
  return GRAINS_OK;
}

extern "C" int grains_get_contact_count(grains_ctx_t* ctx, int32_t* counts, uint64_t n) {
  if (!ctx || !counts) return GRAINS_EINVAL;
  if (n != ctx->n) return fail(ctx, GRAINS_EINVAL, "particle count mismatch");
  GR_HIP(hipStreamSynchronize(ctx->stream));
  GR_HIP(hipMemcpy(counts, ctx->d.contact_count, n * 4, hipMemcpyDeviceToHost));
  return GRAINS_OK;
}

extern "C" int grains_reset_contact_count(grains_ctx_t* ctx) {
  if (!ctx || !ctx->n) return GRAINS_EINVAL;
  launch_fill_u32((uint32_t*)ctx->d.contact_count, ctx->n, 0u, ctx->stream);
  GR_HIP(hipStreamSynchronize(ctx->stream));
  return GRAINS_OK;
}

extern "C" int grains_get_torce(grains_ctx_t* ctx, double* force, double* torque, uint64_t n) {
  if (!ctx) return GRAINS_EINVAL;
  if (n != ctx->n) return fail(ctx, GRAINS_EINVAL, "particle count mismatch");
  GR_HIP(hipStreamSynchronize(ctx->stream));
  std::vector<double> buf(3 * n);
  for (int w = 0; w < 2; ++w) {
    double* dst = w ? torque : force;
    if (!dst) continue;
    GR_HIP(hipMemcpy(buf.data(), w ? ctx->d.last_torque : ctx->d.last_force, 3 * n * 8, hipMemcpyDeviceToHost));
    for (uint64_t i = 0; i < n; ++i)
      for (int k = 0; k < 3; ++k) dst[3 * i + k] = buf[k * n + i];
  }
  return GRAINS_OK;
}

extern "C" int grains_get_stats(grains_ctx_t* ctx, grains_stats_t* st) {
  if (!ctx || !st) return GRAINS_EINVAL;
  *st = ctx->stats;
  return GRAINS_OK;
}

// the shape set rides in the batch kernel's arguments
static bool shapes_in_args(const grains_ctx* ctx) {
  bool in_args = ctx->na_np64.size() <= (size_t)kArgShapes;
  for (size_t k = 0; in_args && k < ctx->na_np64.size(); ++k) in_args = ctx->na_np64[k].kind != GRAINS_POLYHEDRON;
  return in_args;
}

extern "C" int grains_gjk_batch_device(grains_ctx_t* ctx, const uint32_t* sa, const uint32_t* sb, const double* ta,
                                       const double* tb, uint64_t n, double* dist, int32_t* iters, float* ms) {
  if (!ctx || !sa || !sb || !ta || !tb || !dist) return GRAINS_EINVAL;
  if (ctx->shapes.empty()) return fail(ctx, GRAINS_ESTATE, "no shapes");
  // shape tables only (no particles needed)
  const size_t S = ctx->shapes.size();
  const std::vector<ShapeNP<double>>& np64 = ctx->na_np64;
  const std::vector<ShapeNP<float>>& np32 = ctx->na_np32;
  const std::vector<double>& v64 = ctx->na_v64;
  const std::vector<float>& v32 = ctx->na_v32;
  const bool in_args = shapes_in_args(ctx);
  std::vector<void*> tmp;
  ShapeNP<double>* p64 = nullptr;
  ShapeNP<float>* p32 = nullptr;
  double* pv64 = nullptr;
  float* pv32 = nullptr;
  hipStream_t s = ctx->stream;
  int rc;
  // The call comes after what the caller has put on the default stream (the
  // arrays may be its results), as the copies of the tables below do.
  if (in_args) (void)hipStreamSynchronize(nullptr);
  if (!in_args) {
    if ((rc = dalloc(ctx, &p64, S * sizeof(ShapeNP<double>), tmp)) || (rc = dalloc(ctx, &p32, S * sizeof(ShapeNP<float>), tmp)) ||
        (rc = dalloc(ctx, &pv64, v64.size() * 8, tmp)) || (rc = dalloc(ctx, &pv32, v32.size() * 4, tmp))) {
      free_list(tmp);
      return rc;
    }
    (void)hipMemcpy(p64, np64.data(), S * sizeof(ShapeNP<double>), hipMemcpyHostToDevice);
    (void)hipMemcpy(p32, np32.data(), S * sizeof(ShapeNP<float>), hipMemcpyHostToDevice);
    (void)hipMemcpy(pv64, v64.data(), v64.size() * 8, hipMemcpyHostToDevice);
    (void)hipMemcpy(pv32, v32.data(), v32.size() * 4, hipMemcpyHostToDevice);
  }
  const GjkArgs args = {ctx->cfg.flags, ctx->cfg.gjk_rel_tol};
  (void)hipEventRecord(ctx->ev0, s);
  if (in_args && ctx->cfg.precision == GRAINS_FP64)
    launch_gjk_batch_args64(np64.data(), S, sa, sb, ta, tb, n, args, dist, iters, s);
  else if (in_args)
    launch_gjk_batch_args32(np32.data(), S, sa, sb, ta, tb, n, args, dist, iters, s);
  else if (ctx->cfg.precision == GRAINS_FP64)
    launch_gjk_batch64(p64, pv64, sa, sb, ta, tb, n, args, dist, nullptr, nullptr, iters, s);
  else
    launch_gjk_batch32(p32, pv32, sa, sb, ta, tb, n, args, dist, nullptr, nullptr, iters, s);
  (void)hipEventRecord(ctx->ev1, s);
  hipError_t e = hipStreamSynchronize(s);
  float t = 0;
  (void)hipEventElapsedTime(&t, ctx->ev0, ctx->ev1);
  if (ms) *ms = t;
  free_list(tmp);
  if (e != hipSuccess) return fail(ctx, GRAINS_EDEVICE, hipGetErrorString(e));
  return GRAINS_OK;
}

extern "C" int grains_gjk_batch(grains_ctx_t* ctx, const uint32_t* sa, const uint32_t* sb, const double* ta,
                                const double* tb, uint64_t n, double* dist, double* pa, double* pb, int32_t* iters) {
  if (!ctx || !sa || !sb || !ta || !tb || !dist || !n) return GRAINS_EINVAL;
  for (uint64_t k = 0; k < n; ++k)
    if (sa[k] >= ctx->shapes.size() || sb[k] >= ctx->shapes.size())
      return fail(ctx, GRAINS_EINVAL, "shape index out of range");
  std::vector<void*> tmp;
  uint32_t *dsa, *dsb;
  double *dta, *dtb, *dd, *dpa, *dpb;
  int32_t* dit;
  int rc;
  if ((rc = dalloc(ctx, &dsa, n * 4, tmp)) || (rc = dalloc(ctx, &dsb, n * 4, tmp)) ||
      (rc = dalloc(ctx, &dta, n * 96, tmp)) || (rc = dalloc(ctx, &dtb, n * 96, tmp)) ||
      (rc = dalloc(ctx, &dd, n * 8, tmp)) || (rc = dalloc(ctx, &dpa, n * 24, tmp)) ||
      (rc = dalloc(ctx, &dpb, n * 24, tmp)) || (rc = dalloc(ctx, &dit, n * 4, tmp))) {
    free_list(tmp);
    return rc;
  }
  (void)hipMemcpy(dsa, sa, n * 4, hipMemcpyHostToDevice);
  (void)hipMemcpy(dsb, sb, n * 4, hipMemcpyHostToDevice);
  (void)hipMemcpy(dta, ta, n * 96, hipMemcpyHostToDevice);
  (void)hipMemcpy(dtb, tb, n * 96, hipMemcpyHostToDevice);
  // shape tables
  const size_t S = ctx->shapes.size();
  const std::vector<ShapeNP<double>>& np64 = ctx->na_np64;
  const std::vector<ShapeNP<float>>& np32 = ctx->na_np32;
  const std::vector<double>& v64 = ctx->na_v64;
  const std::vector<float>& v32 = ctx->na_v32;
  ShapeNP<double>* p64;
  ShapeNP<float>* p32;
  double* pv64;
  float* pv32;
  if ((rc = dalloc(ctx, &p64, S * sizeof(ShapeNP<double>), tmp)) || (rc = dalloc(ctx, &p32, S * sizeof(ShapeNP<float>), tmp)) ||
      (rc = dalloc(ctx, &pv64, v64.size() * 8, tmp)) || (rc = dalloc(ctx, &pv32, v32.size() * 4, tmp))) {
    free_list(tmp);
    return rc;
  }
  (void)hipMemcpy(p64, np64.data(), S * sizeof(ShapeNP<double>), hipMemcpyHostToDevice);
  (void)hipMemcpy(p32, np32.data(), S * sizeof(ShapeNP<float>), hipMemcpyHostToDevice);
  (void)hipMemcpy(pv64, v64.data(), v64.size() * 8, hipMemcpyHostToDevice);
  (void)hipMemcpy(pv32, v32.data(), v32.size() * 4, hipMemcpyHostToDevice);
  const GjkArgs args = {ctx->cfg.flags, ctx->cfg.gjk_rel_tol};
  (void)hipEventRecord(ctx->ev0, ctx->stream);
  if (ctx->cfg.precision == GRAINS_FP64)
    launch_gjk_batch64(p64, pv64, dsa, dsb, dta, dtb, n, args, dd, dpa, dpb, dit, ctx->stream);
  else
    launch_gjk_batch32(p32, pv32, dsa, dsb, dta, dtb, n, args, dd, dpa, dpb, dit, ctx->stream);
  (void)hipEventRecord(ctx->ev1, ctx->stream);
  hipError_t e = hipStreamSynchronize(ctx->stream);
  if (e == hipSuccess) {
    float t = 0;
    (void)hipEventElapsedTime(&t, ctx->ev0, ctx->ev1);
    ctx->stats.elapsed_ms = t;
  }
  if (e == hipSuccess) {
    (void)hipMemcpy(dist, dd, n * 8, hipMemcpyDeviceToHost);
    if (pa) (void)hipMemcpy(pa, dpa, n * 24, hipMemcpyDeviceToHost);
    if (pb) (void)hipMemcpy(pb, dpb, n * 24, hipMemcpyDeviceToHost);
    if (iters) (void)hipMemcpy(iters, dit, n * 4, hipMemcpyDeviceToHost);
  }
  free_list(tmp);
  if (e != hipSuccess) return fail(ctx, GRAINS_EDEVICE, hipGetErrorString(e));
  return GRAINS_OK;
}

static size_t align256(size_t b) { return (b + 255) & ~size_t(255); }

// grains_gjk_batch_device with the shape tables in `scratch` (through the
// address grains_create looked up) instead of memory allocated per call.
// Every call on one GPU shares that GPU's copy and overwrites the tables it
// uses before its kernel reads them; calls that overlap on one GPU race.
extern "C" int grains_gjk_batch_device_noalloc(grains_ctx_t* ctx, const uint32_t* sa, const uint32_t* sb,
                                               const double* ta, const double* tb, uint64_t n, double* dist,
                                               int32_t* iters, float* ms) {
  if (!ctx || !sa || !sb || !ta || !tb || !dist) return GRAINS_EINVAL;
  if (ctx->shapes.empty()) return fail(ctx, GRAINS_ESTATE, "no shapes");
  if (!ctx->scratch) return fail(ctx, GRAINS_ESTATE, "no scratch address on this context's GPU");
  const bool fp64 = ctx->cfg.precision == GRAINS_FP64;
  const size_t S = ctx->shapes.size();
  const size_t bt = align256(S * (fp64 ? sizeof(ShapeNP<double>) : sizeof(ShapeNP<float>)));
  const size_t bv = fp64 ? ctx->na_v64.size() * sizeof(double) : ctx->na_v32.size() * sizeof(float);
  if (bt + align256(bv) > kScratchBytes)
    return fail(ctx, GRAINS_EINVAL,
                "shape tables of " + std::to_string(bt + align256(bv)) + " bytes exceed the " +
                    std::to_string(kScratchBytes) + " bytes of the allocation-free GJK batch");
  if (ms) *ms = 0.0f;
  if (n == 0) return GRAINS_OK;
  hipStream_t s = ctx->stream;
  unsigned char* tab = ctx->scratch;
  unsigned char* ver = ctx->scratch + bt;
  const bool in_args = shapes_in_args(ctx);
  if (!in_args) {
    GR_HIP(hipMemcpyAsync(tab, fp64 ? (const void*)ctx->na_np64.data() : (const void*)ctx->na_np32.data(),
                          S * (fp64 ? sizeof(ShapeNP<double>) : sizeof(ShapeNP<float>)), hipMemcpyHostToDevice, s));
    GR_HIP(hipMemcpyAsync(ver, fp64 ? (const void*)ctx->na_v64.data() : (const void*)ctx->na_v32.data(), bv,
                          hipMemcpyHostToDevice, s));
  }
  const GjkArgs args = {ctx->cfg.flags, ctx->cfg.gjk_rel_tol};
  GR_HIP(hipEventRecord(ctx->ev0, s));
  if (in_args && fp64)
    launch_gjk_batch_args64(ctx->na_np64.data(), S, sa, sb, ta, tb, n, args, dist, iters, s);
  else if (in_args)
    launch_gjk_batch_args32(ctx->na_np32.data(), S, sa, sb, ta, tb, n, args, dist, iters, s);
  else if (fp64)
    launch_gjk_batch64((const ShapeNP<double>*)tab, (const double*)ver, sa, sb, ta, tb, n, args, dist, nullptr,
                       nullptr, iters, s);
  else
    launch_gjk_batch32((const ShapeNP<float>*)tab, (const float*)ver, sa, sb, ta, tb, n, args, dist, nullptr,
                       nullptr, iters, s);
  GR_HIP(hipGetLastError());
  GR_HIP(hipEventRecord(ctx->ev1, s));
  GR_HIP(hipStreamSynchronize(s));
  float t = 0.0f;
  GR_HIP(hipEventElapsedTime(&t, ctx->ev0, ctx->ev1));
  if (ms) *ms = t;
  return GRAINS_OK;
}

// snapshot layout: u64 n, then pos[3n], quat[4n], vel[3n], omega[3n] (FP64,
// component planes), contact counts[n] (i32)
extern "C" int grains_snapshot(grains_ctx_t* ctx, void* bytes, size_t* size) {
  if (!ctx || !size) return GRAINS_EINVAL;
  const uint64_t n = ctx->n;
  const size_t nh = ctx->d.ab_hist ? 12 * n * 8 : 0;  // the two-step scheme's history
  const size_t need = 8 + 13 * n * 8 + n * 4 + nh;
  if (!bytes) {
    *size = need;
    return GRAINS_OK;
  }
  if (*size < need) return fail(ctx, GRAINS_EINVAL, "snapshot buffer too small");
  GR_HIP(hipStreamSynchronize(ctx->stream));
  char* p = (char*)bytes;
  std::memcpy(p, &n, 8);
  p += 8;
  GR_HIP(hipMemcpy(p, ctx->d.pos, 13 * n * 8, hipMemcpyDeviceToHost));
  p += 13 * n * 8;
  GR_HIP(hipMemcpy(p, ctx->d.contact_count, n * 4, hipMemcpyDeviceToHost));
  p += n * 4;
  if (nh) GR_HIP(hipMemcpy(p, ctx->d.ab_hist, nh, hipMemcpyDeviceToHost));
  *size = need;
  return GRAINS_OK;
}

extern "C" int grains_restore(grains_ctx_t* ctx, const void* bytes, size_t size) {
  if (!ctx || !bytes) return GRAINS_EINVAL;
  const uint64_t n = ctx->n;
  uint64_t n0;
  if (size < 8) return GRAINS_EINVAL;
  std::memcpy(&n0, bytes, 8);
  const size_t nh = ctx->d.ab_hist ? 12 * n * 8 : 0;
  if (n0 != n || size < 8 + 13 * n * 8 + n * 4 + nh) return fail(ctx, GRAINS_EINVAL, "snapshot does not match");
  GR_HIP(hipStreamSynchronize(ctx->stream));
  const char* p = (const char*)bytes + 8;
  GR_HIP(hipMemcpy(ctx->d.pos, p, 13 * n * 8, hipMemcpyHostToDevice));
  p += 13 * n * 8;
  GR_HIP(hipMemcpy(ctx->d.contact_count, p, n * 4, hipMemcpyHostToDevice));
  p += n * 4;
  if (nh) GR_HIP(hipMemcpy(ctx->d.ab_hist, p, nh, hipMemcpyHostToDevice));
  return warm_reset(ctx);
}

// ---- differentiation: the reverse sweep ---------------------------------------------
extern "C" int grains_adjoint_record(grains_ctx_t* ctx, uint32_t checkpoint_every) {
  if (!ctx || checkpoint_every == 0) return GRAINS_EINVAL;
  int rc = finalize(ctx);
  if (rc) return rc;
  if (ctx->cfg.flags & GRAINS_REF_QUIRKS)
    return fail(ctx, GRAINS_EUNSUPPORTED, "the adjoint covers the physics semantics (no REF_QUIRKS)");
  for (uint32_t s : ctx->pshape) {
    const grains_shape_t& h = ctx->shapes[s].s;
    const bool ell = h.kind == GRAINS_SUPERQUADRIC && h.dims[3] == 2.0 && h.dims[4] == 2.0;
    if (h.kind != GRAINS_SPHERE && !ell)
      return fail(ctx, GRAINS_EUNSUPPORTED, "the adjoint covers spheres and ellipsoids (superquadrics n1 = n2 = 2)");
  }
  for (const auto& t : ctx->tables)
    if (t.kr != 0.0) return fail(ctx, GRAINS_EUNSUPPORTED, "the adjoint covers kr = 0 (no rolling resistance)");
  if (ctx->d.gen_obs) return fail(ctx, GRAINS_EUNSUPPORTED, "the adjoint covers Rectangle obstacles");
  if (ctx->cfg.integrator != GRAINS_FIRST_ORDER_EXPLICIT)
    return fail(ctx, GRAINS_EUNSUPPORTED, "the adjoint covers FirstOrderExplicit");
  if (ctx->d.warm)
    return fail(ctx, GRAINS_EUNSUPPORTED, "the adjoint replays steps from checkpoints: no GRAINS_WARM_START");
  // the sweep's buffers are sized by checkpoint_every: drop them
  free_list(ctx->adj_cp);
  free_list(ctx->adj_allocs);
  free_list(ctx->adj_gjk);
  free_list(ctx->adj_log_allocs);
  ctx->adj_log.clear();
  ctx->adj_log_off = false;
  ctx->adj_log_ok = true;
  ctx->ab = AdjBufs{};
  ctx->adj_blk = ctx->adj_save = nullptr;
  ctx->adj_count = nullptr;
  if (!ctx->adj_rec) drop_graph(ctx);  // a recorded step logs its state
  ctx->adj_every = checkpoint_every;
  ctx->adj_steps = 0;
  ctx->adj_rec = true;
  double* cp;
  if ((rc = adj_dalloc(ctx, &cp, 13 * ctx->n * 8, ctx->adj_cp)) || (rc = state_to(ctx, cp))) return rc;
  GR_HIP(hipStreamSynchronize(ctx->stream));
  return GRAINS_OK;
}

extern "C" int grains_adjoint(grains_ctx_t* ctx, const double* dL_dstate, double* dL_dparams, double* dL_dstate0) {
  if (!ctx || !dL_dstate || !dL_dparams) return GRAINS_EINVAL;
  if (!ctx->adj_rec) return fail(ctx, GRAINS_ESTATE, "no recorded trajectory (grains_adjoint_record)");
  const uint64_t n = ctx->n, ecap = ctx->d.ecap, T = ctx->adj_steps, K = ctx->adj_every;
  const uint32_t ntab = (uint32_t)ctx->tables.size();
  hipStream_t s = ctx->stream;
  int rc;
  AdjBufs& a = ctx->ab;
  if (!ctx->adj_save) {
    uint32_t max_obs = 1;
    for (const SimGrid& g : ctx->grids) max_obs = std::max(max_obs, g.obs_end - g.obs_begin);
    auto& L = ctx->adj_allocs;
    if ((rc = adj_dalloc(ctx, &ctx->adj_save, 13 * n * 8, L)) ||
        (rc = adj_dalloc(ctx, &ctx->adj_count, n * 4, L)) || (rc = adj_dalloc(ctx, &a.abar, 13 * n * 8, L)) ||
        (rc = adj_dalloc(ctx, &a.own, 13 * n * 8, L)) || (rc = adj_dalloc(ctx, &a.Fb, 3 * n * 8, L)) ||
        (rc = adj_dalloc(ctx, &a.Mb, 3 * n * 8, L)) || (rc = adj_dalloc(ctx, &a.part_i, ecap * 13 * 8, L)) ||
        (rc = adj_dalloc(ctx, &a.part_j, ecap * 13 * 8, L)) || (rc = adj_dalloc(ctx, &a.entry_theta, ecap * 4 * 8, L)) ||
        (rc = adj_dalloc(ctx, &a.entry_tidx, ecap * 4, L)) || (rc = adj_dalloc(ctx, &a.wall_theta, n * max_obs * 4 * 8, L)) ||
        (rc = adj_dalloc(ctx, &a.wall_tidx, n * max_obs * 4, L)) || (rc = adj_dalloc(ctx, &a.dtheta, (size_t)ntab * 4 * 8, L))) {
      free_list(L);
      free_list(ctx->adj_gjk);
      a = AdjBufs{};
      ctx->adj_save = ctx->adj_blk = nullptr;
      return rc;
    }
    a.max_obs = max_obs;
  }
  // blocks whose steps have to be run again from their checkpoint
  auto logged = [&](uint64_t bb) { return K == 1 || (ctx->adj_log_ok && ctx->adj_log[bb]); };
  for (uint64_t bb = 0; bb * K < T; ++bb)
    if (!logged(bb) && !ctx->adj_blk && (rc = adj_dalloc(ctx, &ctx->adj_blk, K * 13 * n * 8, ctx->adj_allocs))) return rc;
  // the FP64 searches of two passes leave their results for the adjoint of
  // their contacts; in one pass, or without the memory for them, it searches
  // again (the passes can change from one sweep to the next)
  const bool rec = ctx->d.precision == GRAINS_FP64 && ctx->d.split > 0;
  if (rec && !a.gjk) (void)adj_spare(ctx, &a.gjk, ecap * sizeof(GjkRec), ctx->adj_gjk);
  // the state adjoint, rows -> planes
  {
    std::vector<double> planes(13 * n);
    const double* pos = dL_dstate;
    const double* quat = pos + 3 * n;
    const double* vel = quat + 4 * n;
    const double* om = vel + 3 * n;
    for (uint64_t i = 0; i < n; ++i) {
      for (int k = 0; k < 3; ++k) planes[k * n + i] = pos[3 * i + k];
      for (int k = 0; k < 4; ++k) planes[(3 + k) * n + i] = quat[4 * i + k];
      for (int k = 0; k < 3; ++k) planes[(7 + k) * n + i] = vel[3 * i + k];
      for (int k = 0; k < 3; ++k) planes[(10 + k) * n + i] = om[3 * i + k];
    }
    GR_HIP(hipMemcpy(a.abar, planes.data(), 13 * n * 8, hipMemcpyHostToDevice));
  }
  launch_fill_u32((uint32_t*)a.dtheta, (uint64_t)ntab * 8, 0u, s);
  if ((rc = state_to(ctx, ctx->adj_save))) return rc;
  GR_HIP(hipMemcpyAsync(ctx->adj_count, ctx->d.contact_count, n * 4, hipMemcpyDeviceToDevice, s));
  const bool prof = ctx->profiling;
  ctx->profiling = false;
  // every step below sets its state: its lists are built for it alone
  const bool skin = ctx->d.skin != 0;
  if (skin && (rc = use_skin(ctx, false))) return rc;
  ctx->lists_ok = false;
  ctx->d.keep_torce = 1;
  launch_run_begin(ctx->d, 0u, true, s);
  ctx->d.gjk_rec = rec ? a.gjk : nullptr;
  const uint64_t nblocks = (T + K - 1) / K;
  for (uint64_t bb = nblocks; bb-- > 0;) {
    const uint64_t t0 = bb * K, t1 = std::min(t0 + K, T);
    double* first = (double*)ctx->adj_cp[bb];
    double* states = logged(bb) ? ctx->adj_log[bb] : ctx->adj_blk;
    if (!logged(bb)) {
      if ((rc = state_from(ctx, first))) break;
      for (uint64_t t = t0; t < t1 && !rc; ++t) {
        if ((rc = state_to(ctx, states + (t - t0) * 13 * n))) break;
        enqueue_step(ctx, true);
      }
    }
    for (uint64_t t = t1; t-- > t0 && !rc;) {
      double* st = t == t0 ? first : states + (t - t0) * 13 * n;
      if ((rc = state_from(ctx, st))) break;
      enqueue_step(ctx, true);  // entries, contact flags, force and torque of step t
      a.state = st;
      launch_adjoint_step(ctx->d, a, ntab, s);
    }
    if (rc) break;
  }
  ctx->profiling = prof;
  ctx->d.keep_torce = 0;
  ctx->d.gjk_rec = nullptr;
  int rc2 = state_from(ctx, ctx->adj_save);
  if (skin && !rc2) rc2 = use_skin(ctx, true);
  if (rc) return rc;
  if (rc2) return rc2;
  GR_HIP(hipMemcpyAsync(ctx->d.contact_count, ctx->adj_count, n * 4, hipMemcpyDeviceToDevice, s));
  GR_HIP(hipGetLastError());
  GR_HIP(hipStreamSynchronize(s));
  GR_HIP(hipMemcpy(dL_dparams, a.dtheta, (size_t)ntab * 4 * 8, hipMemcpyDeviceToHost));
  if (dL_dstate0) {
    std::vector<double> planes(13 * n);
    GR_HIP(hipMemcpy(planes.data(), a.abar, 13 * n * 8, hipMemcpyDeviceToHost));
    double* pos = dL_dstate0;
    double* quat = pos + 3 * n;
    double* vel = quat + 4 * n;
    double* om = vel + 3 * n;
    for (uint64_t i = 0; i < n; ++i) {
      for (int k = 0; k < 3; ++k) pos[3 * i + k] = planes[k * n + i];
      for (int k = 0; k < 4; ++k) quat[4 * i + k] = planes[(3 + k) * n + i];
      for (int k = 0; k < 3; ++k) vel[3 * i + k] = planes[(7 + k) * n + i];
      for (int k = 0; k < 3; ++k) om[3 * i + k] = planes[(10 + k) * n + i];
    }
  }
  return GRAINS_OK;
}
