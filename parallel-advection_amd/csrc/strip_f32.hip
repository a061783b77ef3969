// Strip kernels, FP32 storage: fused sums, FP64 between the steps of a pass.
#include "strip_launch.hpp"

namespace bkma {

bkma_status launch_strip_f32(const TileShape &sh, const TileArgs &a, void *data, void *halo, hipStream_t s) {
    return launch_strip<float, true, false>(sh, a, data, halo, s);
}

bkma_status launch_strip_group_f32(const TileGroup &g, int ns, hipStream_t s) {
    return launch_strip_group<float, true, false>(g, ns, s);
}

}  // namespace bkma
