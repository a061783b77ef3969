// Strip kernels, FP32 storage: fused sums, rounded to FP32 after every step.
#include "strip_launch.hpp"

namespace bkma {

bkma_status launch_strip_f32_round(const TileShape &sh, const TileArgs &a, void *data, void *halo, hipStream_t s) {
    return launch_strip<float, true, true>(sh, a, data, halo, s);
}

bkma_status launch_strip_group_f32_round(const TileGroup &g, int ns, hipStream_t s) {
    return launch_strip_group<float, true, true>(g, ns, s);
}

}  // namespace bkma
