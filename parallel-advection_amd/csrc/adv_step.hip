// One advection step of a whole array for the reference's executors
// (bkma_adv_run): the values do not depend on how an executor cuts the array
// into work-groups, so a call whose one batch covers the array takes the
// kernel that reads and writes every cell once.
//
// The executors evaluate the foot and lag_basis at every cell and index with
// 64-bit divisions; on [2048][1024][64] FP64 that is 38 Gcell/s, held by the
// VALU.  Here
//  - FP64 arrays of many columns stream through registers
//    (adv_step_column_kernel: the column-pair kernel's one-step form, its
//    coefficients one row per lane of a wavefront): 0.43 ms = 5.0 TB/s;
//  - other lines go through the LDS tiles of adv_tile.hpp with one step per
//    pass, one foot per row and four columns: 0.60 ms on that shape.
#include <algorithm>
#include <climits>

#include "adv_pair.hpp"
#include "adv_step.hpp"
#include "adv_tile.hpp"

namespace bkma {

namespace {

constexpr int kStepRows = 8;   // head rows per wave: 6 of the pair form, 7 of the ring form
constexpr int kStepWaves = 4;  // wavefronts per work-group (no barrier between them)

}  // namespace

// A wavefront first finds the shifts of its slab's rows.  One shift for all
// rows (almost every slab) runs the six-tap body of that shift; rows that
// round to two sides run the ring of adv_stream.hpp, which reads each row's
// own six taps (the seven-tap body would multiply a cell that the reference
// does not read by zero).
template <int VEC>
__global__ __launch_bounds__(64 * kStepWaves) void adv_step_column_kernel(double *__restrict__ data, StreamArgs a) {
    __shared__ double head_lds[kStepWaves][kStepRows][64 * VEC];
    const int lane = threadIdx.x & 63;
    const int wv = wave_uniform((int)(threadIdx.x >> 6));
    const i64 unit = (i64)blockIdx.x * kStepWaves + wv;
    if (unit >= a.total_units) return;
    const i64 i0 = unit / a.tiles_per_slab, tile = unit - i0 * a.tiles_per_slab;
    const int n1 = (int)a.p.n1, half = n1 / 2;
    int lo = INT_MAX, hi = INT_MIN;
    for (int row = lane; row < n1; row += 64) {
        double d_prev1;
        int d = row - adv_foot(a.p, (int)i0, row, d_prev1);
        if (d > half) d -= n1;
        if (d < -half) d += n1;
        lo = min(lo, d);
        hi = max(hi, d);
    }
#pragma unroll
    for (int m = 32; m > 0; m >>= 1) {
        lo = min(lo, __shfl_xor(lo, m));
        hi = max(hi, __shfl_xor(hi, m));
    }
    lo = wave_uniform(lo);
    hi = wave_uniform(hi);
    if (lo == hi)
        pair_dispatch<double, double, VEC, 14, 1, true, false, 6, -3, 3>(lo, data, a, i0, tile, lane, head_lds[wv]);
    else
        stream_unit<double, double, VEC, 4, 7, 1, true>(data, a, unit, lane, head_lds[wv]);
}

namespace {

// Shapes of the register form: whole 128-column (64 below 128) tiles, shifts
// within [-3, 3] up to the rounding of the feet (tile_shifts; the kernel has no
// body for any other), and wavefronts enough to fill the GPU.  Time of the tiles
// over it, one FP64 step of [n0][1000][n2]: n2 = 64: 512 slabs 0.78, 1024
// 1.23; n2 = 128: 256 slabs 0.70, 512 1.23; [n0][3000][64]: 256 slabs 1.1.
bool column_form(const AdvDev &p, const void *data) {
    const i64 width = p.n2 >= 128 ? 128 : 64;
    if (p.n2 % width != 0 || p.n1 < 64 || p.n1 > (1 << 20)) return false;
    if (width == 128 && reinterpret_cast<uintptr_t>(data) % 16 != 0) return false;
    if (p.n0 * (p.n2 / 64) < (p.n1 > 2500 ? 256 : 1024) || p.n0 * (p.n2 / width) > 0x7fffffffLL) return false;
    double lo0, hi0, lo1, hi1;
    tile_shifts(p, 0, lo0, hi0);
    tile_shifts(p, p.n0 - 1, lo1, hi1);
    return std::min(lo0, lo1) >= -3.0 && std::max(hi0, hi1) <= 3.0;
}

template <int VEC> bkma_status launch_column(const AdvDev &p, double *data, hipStream_t s) {
    StreamArgs a{};
    a.p = p;
    a.tiles_per_slab = p.n2 / (64 * VEC);
    a.total_units = p.n0 * a.tiles_per_slab;
    hipLaunchKernelGGL(adv_step_column_kernel<VEC>, dim3((unsigned)ceil_div((u64)a.total_units, kStepWaves)),
                       dim3(64 * kStepWaves), 0, s, data, a);
    return check_launch("adv_step_column_kernel");
}

// The tile shapes of the last sizes that this thread stepped (a time loop
// calls with one size; choosing a shape compares some tens of them).
struct StepShape {
    i64 n0 = 0, n1 = 0, n2 = 0;
    u64 esz = 0, lds_max = 0;
    bool fits = false;
    TileShape tile;
};

const StepShape &step_shape(const AdvDev &p, u64 esz, u64 lds_max) {
    static thread_local StepShape kept[16];
    StepShape &k = kept[(u64)(p.n0 * 7 + p.n1 * 3 + p.n2 + (i64)esz) % 16];
    if (k.n0 != p.n0 || k.n1 != p.n1 || k.n2 != p.n2 || k.esz != esz || k.lds_max != lds_max) {
        k.n0 = p.n0;
        k.n1 = p.n1;
        k.n2 = p.n2;
        k.esz = esz;
        k.lds_max = lds_max;
        bkma_adv_params q{};
        q.n0 = (u64)p.n0;
        q.n1 = (u64)p.n1;
        q.n2 = (u64)p.n2;
        k.fits = p.n1 <= kTileRows * kTileThreads && tile_shape(q, 0, q.n0, esz, 1, lds_max, &k.tile, true);
    }
    return k;
}

}  // namespace

bkma_status adv_step_whole(const AdvDev &p, bkma_dtype dt, void *data, hipStream_t s, bool *done) {
    *done = false;
    if (p.n1 < 16 || !tile_covers(p)) return BKMA_OK;
    if (dt == BKMA_F64 && column_form(p, data)) {
        *done = true;
        return p.n2 >= 128 ? launch_column<2>(p, (double *)data, s) : launch_column<1>(p, (double *)data, s);
    }
    u64 lds_max = 0;
    BKMA_TRY(lds_limit_bytes(&lds_max));
    const StepShape &k = step_shape(p, dt == BKMA_F64 ? 8 : 4, lds_max);
    if (!k.fits) return BKMA_OK;
    *done = true;
    TileShape sh = k.tile;
    sh.a.p = p;
    // the executors' sums are separately rounded whatever the storage
    return launch_tile(sh, dt, false, false, data, nullptr, 1, s);
}

}  // namespace bkma
