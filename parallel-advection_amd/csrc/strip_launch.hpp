// Kernels and launchers of the strip form for one arithmetic (strip_f64.hip,
// strip_f32.hip, strip_f32_round.hip instantiate them, so that they compile in
// parallel).
#pragma once

#include "adv_strip.hpp"

namespace bkma {

template <class T, bool FUSED, bool RND, int E, bool WRAP>
__global__ __launch_bounds__(kStripMaxThreads) void adv_strip_kernel(T *__restrict__ data, const T *__restrict__ halo,
                                                                     TileArgs a) {
    extern __shared__ __align__(16) unsigned char tile_lds[];
    strip_unit<T, FUSED, RND, E, WRAP>(data, halo, a, tile_of_block(blockIdx.x, a.units, a.nct),
                                       reinterpret_cast<double *>(tile_lds));
}

template <class T, bool FUSED, bool RND, int E, bool WRAP>
__global__ __launch_bounds__(kStripMaxThreads) void adv_strip_group_kernel(const TileProblem *__restrict__ tab,
                                                                           int count, int ns) {
    extern __shared__ __align__(16) unsigned char tile_lds[];
    const TileProblem &pr = tab[problem_of_block<&TileProblem::first>(tab, count, blockIdx.x)];
    TileArgs a = pr.a;
    a.ns = ns;
    strip_unit<T, FUSED, RND, E, WRAP>((T *)pr.data, (const T *)pr.halo, a,
                                       tile_of_block((i64)blockIdx.x - pr.first, a.units, a.nct),
                                       reinterpret_cast<double *>(tile_lds));
}

template <class T, bool FUSED, bool RND, int E, bool WRAP>
bkma_status launch_strip_e(const TileShape &sh, const TileArgs &a, void *data, void *halo, hipStream_t s) {
    static std::atomic<unsigned> done{0};
    auto k = adv_strip_kernel<T, FUSED, RND, E, WRAP>;
    BKMA_TRY(allow_lds(k, done));
    hipLaunchKernelGGL(k, dim3((unsigned)a.units), dim3((unsigned)sh.threads), (size_t)sh.lds_bytes, s, (T *)data,
                       (const T *)halo, a);
    return check_launch("adv_strip_kernel");
}

template <class T, bool FUSED, bool RND, int E, bool WRAP>
bkma_status launch_strip_group_e(const TileGroup &g, int ns, hipStream_t s) {
    static std::atomic<unsigned> done{0};
    auto k = adv_strip_group_kernel<T, FUSED, RND, E, WRAP>;
    BKMA_TRY(allow_lds(k, done));
    hipLaunchKernelGGL(k, dim3((unsigned)g.units), dim3((unsigned)g.threads), (size_t)g.lds_bytes, s,
                       (const TileProblem *)g.table, g.count, ns);
    return check_launch("adv_strip_group_kernel");
}

template <class T, bool FUSED, bool RND>
bkma_status launch_strip(const TileShape &sh, const TileArgs &a, void *data, void *halo, hipStream_t s) {
    if (!sh.wrap) return launch_strip_e<T, FUSED, RND, kStripSegE, false>(sh, a, data, halo, s);
    if (sh.e == 8) return launch_strip_e<T, FUSED, RND, 8, true>(sh, a, data, halo, s);
    if (sh.e == 6) return launch_strip_e<T, FUSED, RND, 6, true>(sh, a, data, halo, s);
    return launch_strip_e<T, FUSED, RND, 4, true>(sh, a, data, halo, s);
}

template <class T, bool FUSED, bool RND> bkma_status launch_strip_group(const TileGroup &g, int ns, hipStream_t s) {
    if (!g.wrap) return launch_strip_group_e<T, FUSED, RND, kStripSegE, false>(g, ns, s);
    if (g.e == 8) return launch_strip_group_e<T, FUSED, RND, 8, true>(g, ns, s);
    if (g.e == 6) return launch_strip_group_e<T, FUSED, RND, 6, true>(g, ns, s);
    return launch_strip_group_e<T, FUSED, RND, 4, true>(g, ns, s);
}

}  // namespace bkma
