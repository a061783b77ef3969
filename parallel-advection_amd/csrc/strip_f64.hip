// Strip kernels, FP64 storage: separately rounded sums.
#include "strip_launch.hpp"

namespace bkma {

bkma_status launch_strip_f64(const TileShape &sh, const TileArgs &a, void *data, void *halo, hipStream_t s) {
    return launch_strip<double, false, false>(sh, a, data, halo, s);
}

bkma_status launch_strip_group_f64(const TileGroup &g, int ns, hipStream_t s) {
    return launch_strip_group<double, false, false>(g, ns, s);
}

}  // namespace bkma
