// gr_narrow32.hip -- FP32-mixed narrow phase (GJK, support maps, Hooke in
// FP32, relative frames taken in FP64), FP64 accumulation and integration.
#include <algorithm>

#include "gr_narrow.hpp"

namespace gr {

void launch_narrow32(const DevScene& d, int pass, hipStream_t s) {
  const bool sv = !(d.flags & GRAINS_REF_QUIRKS);
  const bool two = sv && d.split > 0;
  const bool warm = sv && d.warm;
  const dim3 grid(d.narrow_blocks), block(d.block);
  // The complete pass: no more threads than are resident at once, 512 a CU
  // whatever the block's size: more blocks, most with nothing to do, queue
  // behind the integration's (10^6 superquadrics at rest, 8 blocks per CU and 2:
  // 0.360 and 0.352 ms a step; agitated beds and 64 ensembles within 1 %).  The
  // single pass likewise, its waves packing the list.
  const dim3 cg(std::min(grid.x, (unsigned)cu_count() * 2 * (unsigned)(kBlock / d.block)));
  if (pass == 0) {
    if (two && warm) {
      hipLaunchKernelGGL((k_screen<float, true>), grid, block, 0, s, d);
    } else if (two) {
      hipLaunchKernelGGL((k_screen<float, false>), grid, block, 0, s, d);
    } else if (warm) {
      hipLaunchKernelGGL((k_narrow<float, true, true, true>), cg, block, 0, s, d);
    } else if (sv) {
      hipLaunchKernelGGL((k_narrow<float, true, true>), cg, block, 0, s, d);
    } else {
      launch_narrow_ref<float>(d, s);
    }
  } else if (two && warm) {
    hipLaunchKernelGGL((k_complete<float, true>), cg, block, 0, s, d);
  } else if (two) {
    hipLaunchKernelGGL((k_complete<float, false>), cg, block, 0, s, d);
  }
}
void launch_integrate32(const DevScene& d, hipStream_t s, int part) { launch_integrate_t<float>(d, s, part); }
void launch_gjk_batch_args32(const ShapeNP<float>* shapes, size_t count, const uint32_t* sa, const uint32_t* sb,
                            const double* ta, const double* tb, uint64_t n, GjkArgs args, double* dist,
                            int32_t* iters, hipStream_t s) {
  launch_gjk_batch_args_t<float>(shapes, count, sa, sb, ta, tb, n, args, dist, iters, s);
}
void launch_gjk_batch32(const ShapeNP<float>* shapes, const float* verts, const uint32_t* sa,
                        const uint32_t* sb, const double* ta, const double* tb, uint64_t n, GjkArgs args,
                        double* dist, double* pa, double* pb, int32_t* iters, hipStream_t s) {
  const dim3 grid((unsigned)((n + kBlock - 1) / kBlock));
  if (args.flags & GRAINS_REF_QUIRKS)
    hipLaunchKernelGGL((k_gjk_batch<float, false>), grid, dim3(kBlock), 0, s, shapes, verts, sa, sb, ta, tb, n,
                       args, dist, pa, pb, iters);
  else
    hipLaunchKernelGGL((k_gjk_batch<float, true>), grid, dim3(kBlock), 0, s, shapes, verts, sa, sb, ta, tb, n,
                       args, dist, pa, pb, iters);
}

}  // namespace gr
