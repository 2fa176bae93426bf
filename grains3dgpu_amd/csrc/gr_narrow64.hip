// gr_narrow64.hip -- FP64 ("plain") narrow phase, integration, GJK batch and
// the FP64 re-run used by the FP32-mixed path.  Built with
// -ffp-contract=off so every product and sum rounds as in the reference CPU
// code (and the oracle).
#include <algorithm>

#include "gr_search.hpp"

namespace gr {

// The FP32-mixed path's FP64 re-runs under the reference semantics, one lane
// per entry from scratch (physics semantics: k_search64).
__global__ void __launch_bounds__(kBlock) k_refine64_ref(DevScene d) {
  const uint32_t cnt = *d.refine_count;
  const uint64_t stride = (uint64_t)gridDim.x * blockDim.x;
  uint32_t c_it = 0, c_maxit = 0;
  for (uint64_t k = (uint64_t)blockIdx.x * blockDim.x + threadIdx.x; k < cnt; k += stride) {
    const uint32_t e = d.refine_list[k];
    NpStats st = {0u, 0};
    PairRes<double> r;
    const uint32_t flag = pair_force<double, double, false>(d, d.pair_i[e], d.pair_j[e], r, st, e);
    if (flag & kFlagContact) {
      if (d.res64) {
        ((PairRes<double>*)d.pair_res)[e] = r;
      } else {
        PairRes<float> q;
#pragma unroll
        for (int k3 = 0; k3 < 3; ++k3) q.f[k3] = (float)r.f[k3], q.m[k3] = (float)r.m[k3];
        ((PairRes<float>*)d.pair_res)[e] = q;
      }
    }
    d.pair_flag[e] = flag | kFlagRefine;
    c_it += st.iters;
    c_maxit = c_maxit > (uint32_t)st.iters ? c_maxit : (uint32_t)st.iters;
  }
  count_add(d.counters, kCntRefIters, c_it);
  count_max(d.counters, kCntRefMaxIters, c_maxit);
}

// One narrow pass in FP64 under the physics semantics: the entries that pass the
// prefilter, queued for the complete pass.  The lists hold
// their skin's pairs too, a quarter to a third of the entries; the others,
// searched in the lanes they stand in, take as many waves as the list has, not
// as the step has candidates.  ms a step with lists built for every step,
// entries where they stand, queued: 40,000 touching superquadrics 3.67,
// 5.25, 3.52, 8,191 1.36, 1.28, 1.23, 300,000 loose ones 1.00, 1.07, 0.91.
__global__ void __launch_bounds__(kBlock) k_filter(DevScene d) {
  if (!step_begin(d)) return;
  __shared__ DeferLds L;
  uint32_t nq = 0, c_cand = 0;
  const uint32_t E = d.entry_off[d.n], lane = __lane_id();
  const bool outside = d.nl[kNlOutside] != 0;
  const uint64_t stride = (uint64_t)gridDim.x * blockDim.x;
  // whole waves take turns (the queue appends are wave-wide)
  for (uint64_t e = (uint64_t)blockIdx.x * blockDim.x + threadIdx.x; e - lane < E; e += stride) {
    bool cand = false;
    if (e < E) {
      const uint32_t si = d.pair_i[e], sj = d.pair_j[e];
      const PoseRec pi = d.pk[si], pj = d.pk[sj];
      cand = is_candidate(d.grids[pi.sim], V3<double>{pi.x, pi.y, pi.z}, V3<double>{pj.x, pj.y, pj.z}, d.rcs[si],
                          d.rcs[sj], outside);
      if (!cand) d.pair_flag[e] = 0u;
      c_cand += cand;
    }
    defer_push(d, L, nq, cand, (uint32_t)e);
  }
  defer_flush(d, L, nq);
  count_add(d.counters, kCntCandidates, c_cand);
}
// One wave per block, two per SIMD (the registers' limit).
template <int MODE>
static void launch_search64(const DevScene& d, hipStream_t s) {
  hipLaunchKernelGGL(k_search64<MODE>, dim3((unsigned)cu_count() * 8), dim3(64), 0, s, d);
}

void launch_narrow64(const DevScene& d, int pass, hipStream_t s) {
  const bool sv = !(d.flags & GRAINS_REF_QUIRKS);
  const bool two = d.split > 0;
  if (d.balls) {
    if (pass == 0) hipLaunchKernelGGL(k_narrow_balls<double>, dim3(d.narrow_blocks), dim3(d.block), 0, s, d);
  } else if (pass == 0) {
    if (two && sv)
      hipLaunchKernelGGL((k_screen<double, false>), dim3(d.narrow_blocks), dim3(d.block), 0, s, d);
    else if (two)
      hipLaunchKernelGGL((k_screen<double, false, false>), dim3(d.narrow_blocks), dim3(d.block), 0, s, d);
    else if (sv) {
      hipLaunchKernelGGL(k_filter, dim3(d.narrow_blocks), dim3(d.block), 0, s, d);
      hipLaunchKernelGGL((k_complete<double, false>), dim3(d.narrow_blocks), dim3(d.block), 0, s, d);
    } else {
      launch_narrow_ref<double>(d, s);
    }
  } else if (two && sv) {
    launch_search64<0>(d, s);
  } else if (two) {
    hipLaunchKernelGGL((k_complete<double, false, false>), dim3(d.narrow_blocks), dim3(d.block), 0, s, d);
  }
}
void launch_refine64(const DevScene& d, hipStream_t s) {
  if (d.flags & GRAINS_REF_QUIRKS)
    hipLaunchKernelGGL(k_refine64_ref, dim3(d.narrow_blocks / 4 + 1), dim3(kBlock), 0, s, d);
  else
    launch_search64<1>(d, s);
}
void launch_integrate64(const DevScene& d, hipStream_t s, int part) { launch_integrate_t<double>(d, s, part); }
void launch_gjk_batch_args64(const ShapeNP<double>* shapes, size_t count, const uint32_t* sa, const uint32_t* sb,
                            const double* ta, const double* tb, uint64_t n, GjkArgs args, double* dist,
                            int32_t* iters, hipStream_t s) {
  launch_gjk_batch_args_t<double>(shapes, count, sa, sb, ta, tb, n, args, dist, iters, s);
}
void launch_gjk_batch64(const ShapeNP<double>* shapes, const double* verts, const uint32_t* sa,
                        const uint32_t* sb, const double* ta, const double* tb, uint64_t n, GjkArgs args,
                        double* dist, double* pa, double* pb, int32_t* iters, hipStream_t s) {
  const dim3 grid((unsigned)((n + kBlock - 1) / kBlock));
  if (args.flags & GRAINS_REF_QUIRKS)
    hipLaunchKernelGGL((k_gjk_batch<double, false>), grid, dim3(kBlock), 0, s, shapes, verts, sa, sb, ta, tb, n,
                       args, dist, pa, pb, iters);
  else
    hipLaunchKernelGGL((k_gjk_batch<double, true>), grid, dim3(kBlock), 0, s, shapes, verts, sa, sb, ta, tb, n,
                       args, dist, pa, pb, iters);
}

}  // namespace gr
