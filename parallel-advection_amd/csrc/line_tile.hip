// Kernels, launch shapes and launchers of the LDS tile form with register
// coefficients (adv_tile.hpp).
#include <algorithm>
#include <atomic>
#include <cmath>

#include "adv_tile.hpp"

namespace bkma {

// Consecutive tiles of one memory line (the column tiles of a slab) on one
// XCD: work-groups go to the 8 XCDs in turn.
__device__ __forceinline__ i64 tile_of_block(i64 b, i64 units, int nct) {
    const i64 per = units / 8;
    return nct > 1 && b < per * 8 ? (b % 8) * per + b / 8 : b;
}

template <class T, bool FUSED, bool RND, int V, bool WRAP>
__global__ __launch_bounds__(kTileThreads) void adv_tile_kernel(T *__restrict__ data, const T *__restrict__ halo,
                                                                TileArgs a) {
    extern __shared__ __align__(16) unsigned char tile_lds[];
    tile_unit<T, FUSED, RND, V, WRAP>(data, halo, a, tile_of_block(blockIdx.x, a.units, a.nct),
                                      reinterpret_cast<double *>(tile_lds));
}

template <class T>
__global__ void tile_snapshot_kernel(const T *__restrict__ data, T *__restrict__ halo, TileArgs a) {
    tile_snapshot_unit(data, halo, a, blockIdx.x);
}

// The last problem whose first work-group is not past b.
template <i64 TileProblem::*FIRST> __device__ __forceinline__ int problem_of_block(const TileProblem *tab, int count, i64 b) {
    int lo = 0, hi = count;
    while (hi - lo > 1) {
        const int mid = (lo + hi) / 2;
        if (tab[mid].*FIRST <= b) lo = mid;
        else hi = mid;
    }
    return lo;
}

template <class T, bool FUSED, bool RND, int V, bool WRAP>
__global__ __launch_bounds__(kTileThreads) void adv_tile_group_kernel(const TileProblem *__restrict__ tab, int count,
                                                                      int ns) {
    extern __shared__ __align__(16) unsigned char tile_lds[];
    const TileProblem &pr = tab[problem_of_block<&TileProblem::first>(tab, count, blockIdx.x)];
    TileArgs a = pr.a;
    a.ns = ns;
    tile_unit<T, FUSED, RND, V, WRAP>((T *)pr.data, (const T *)pr.halo, a,
                                      tile_of_block((i64)blockIdx.x - pr.first, a.units, a.nct),
                                      reinterpret_cast<double *>(tile_lds));
}

template <class T>
__global__ void tile_group_snapshot_kernel(const TileProblem *__restrict__ tab, int count, int ns) {
    const TileProblem &pr = tab[problem_of_block<&TileProblem::first_halo>(tab, count, blockIdx.x)];
    TileArgs a = pr.a;
    a.ns = ns;
    tile_snapshot_unit((const T *)pr.data, (T *)pr.halo, a, (i64)blockIdx.x - pr.first_halo);
}

namespace {

// Allows the whole LDS to the kernel, once per device.
template <class K> hipError_t allow_lds(K kernel, std::atomic<unsigned> &done, u64 bytes) {
    int dev = 0;
    const hipError_t e = hipGetDevice(&dev);
    if (e != hipSuccess) return e;
    const unsigned bit = 1u << (dev & 31);
    if (done.load(std::memory_order_relaxed) & bit) return hipSuccess;
    const hipError_t r =
        hipFuncSetAttribute((const void *)kernel, hipFuncAttributeMaxDynamicSharedMemorySize, (int)bytes);
    if (r == hipSuccess) done.fetch_or(bit, std::memory_order_relaxed);
    return r;
}

template <class T, bool FUSED, bool RND, int V, bool WRAP>
bkma_status launch(const TileShape &sh, const TileArgs &a, void *data, void *halo, hipStream_t s) {
    static std::atomic<unsigned> done{0};
    auto k = adv_tile_kernel<T, FUSED, RND, V, WRAP>;
    u64 lds_max = 0;
    BKMA_TRY(lds_limit_bytes(&lds_max));
    BKMA_HIP_TRY(allow_lds(k, done, lds_max));
    hipLaunchKernelGGL(k, dim3((unsigned)a.units), dim3((unsigned)sh.threads), (size_t)sh.lds_bytes, s, (T *)data,
                       (const T *)halo, a);
    return check_launch("adv_tile_kernel");
}

template <class T, bool FUSED, bool RND>
bkma_status launch_v(const TileShape &sh, const TileArgs &a, void *data, void *halo, hipStream_t s) {
    if (sh.wrap) {
        if (sh.v == 1) return launch<T, FUSED, RND, 1, true>(sh, a, data, halo, s);
        if (sh.v == 2) return launch<T, FUSED, RND, 2, true>(sh, a, data, halo, s);
        return launch<T, FUSED, RND, 4, true>(sh, a, data, halo, s);
    }
    const i64 groups = a.p.n0 * a.nseg;
    const unsigned nt = (i64)a.hrows * a.p.n2 >= 512 ? 256 : 64;
    hipLaunchKernelGGL(tile_snapshot_kernel<T>, dim3((unsigned)groups), dim3(nt), 0, s, (const T *)data, (T *)halo, a);
    BKMA_TRY(check_launch("tile_snapshot_kernel"));
    if (sh.v == 1) return launch<T, FUSED, RND, 1, false>(sh, a, data, halo, s);
    if (sh.v == 2) return launch<T, FUSED, RND, 2, false>(sh, a, data, halo, s);
    return launch<T, FUSED, RND, 4, false>(sh, a, data, halo, s);
}

template <class T, bool FUSED, bool RND, int V, bool WRAP>
bkma_status launch_group(const TileGroup &g, int ns, hipStream_t s) {
    static std::atomic<unsigned> done{0};
    auto k = adv_tile_group_kernel<T, FUSED, RND, V, WRAP>;
    u64 lds_max = 0;
    BKMA_TRY(lds_limit_bytes(&lds_max));
    BKMA_HIP_TRY(allow_lds(k, done, lds_max));
    hipLaunchKernelGGL(k, dim3((unsigned)g.units), dim3((unsigned)g.threads), (size_t)g.lds_bytes, s,
                       (const TileProblem *)g.table, g.count, ns);
    return check_launch("adv_tile_group_kernel");
}

template <class T, bool FUSED, bool RND> bkma_status launch_group_v(const TileGroup &g, int ns, hipStream_t s) {
    if (g.wrap) {
        if (g.v == 1) return launch_group<T, FUSED, RND, 1, true>(g, ns, s);
        if (g.v == 2) return launch_group<T, FUSED, RND, 2, true>(g, ns, s);
        return launch_group<T, FUSED, RND, 4, true>(g, ns, s);
    }
    hipLaunchKernelGGL(tile_group_snapshot_kernel<T>, dim3((unsigned)g.halo_units), dim3(256), 0, s,
                       (const TileProblem *)g.table, g.count, ns);
    BKMA_TRY(check_launch("tile_group_snapshot_kernel"));
    if (g.v == 1) return launch_group<T, FUSED, RND, 1, false>(g, ns, s);
    if (g.v == 2) return launch_group<T, FUSED, RND, 2, false>(g, ns, s);
    return launch_group<T, FUSED, RND, 4, false>(g, ns, s);
}

unsigned magic(u64 d) { return d > 1 ? (unsigned)((((u64)1 << 32) + d - 1) / d) : 0; }

// Plane pitch of at least `rows` doubles: the columns of a row are written by
// neighbouring lanes, so their planes start 32/cb doubles apart modulo the 64
// banks.
int plane_pitch(int rows, int cb) {
    if (cb <= 1) return rows;
    int c2 = 1;
    while (c2 < cb) c2 *= 2;
    const int want = c2 >= 32 ? 1 : 32 / c2;
    return rows + ((want - rows) % 32 + 32) % 32;
}

}  // namespace

bool tile_shape(const bkma_adv_params &p, u64 elem_size, int ns, u64 lds_max, TileShape *out, bool whole_only) {
    if (p.n1 < 16 || p.n0 == 0 || p.n2 == 0) return false;
    // Threads per work-group.  Whole lines: work-groups of four wavefronts,
    // five to a CU, keep the LDS and the VALU busy at different times
    // ([2048][1024][64] FP64, 20 steps: 1436 Gcell/s with 205 threads, 1290
    // with 410).  Segments: longer ones have fewer halo rows.
    constexpr int kWhole = 256, kSegment = 512;
    const u64 n0 = p.n0, n1 = p.n1, n2 = p.n2;
    TileShape sh;
    TileArgs &a = sh.a;
    a.p = make_adv_dev(p);
    a.sb = 1;
    a.nseg = 1;
    a.mn1 = magic(n1);
    auto bytes = [&](int planes, int pitch, int v) { return (u64)planes * pitch * 8 * (v == 1 ? 2 : 1); };
    const u64 rt_line = ceil_div(n1, kTileRows);
    bool whole = false;  // *out holds a whole-line tile
    if (rt_line <= (u64)kTileThreads) {
        // Whole lines.  Of the column widths that fit, the one that keeps the
        // most threads busy: columns that divide n2, whole wavefronts, and
        // several work-groups' worth of wavefronts per CU.
        const int rt = (int)rt_line;
        double best = 0;
        for (int v = n2 >= 3 ? 4 : (int)n2; v >= 1; v /= 2) {
            for (int ct = 1; (ct == 1 || rt * ct <= kWhole) && (u64)(ct - 1) * v < n2; ++ct) {
                const int cols = (int)std::min<u64>((u64)ct * v, n2);
                const int pitch = plane_pitch((int)n1 + kTileGhost, cols);
                for (int sb = 1; sb == 1 || ((u64)cols == n2 && rt * ct * sb <= kWhole && (u64)sb <= n0); ++sb) {
                    const u64 b = bytes(sb * cols, pitch, v);
                    if (b > lds_max) break;
                    const u64 units = ceil_div(n0, (u64)sb) * ceil_div(n2, (u64)cols);
                    if (units > 0x7fffffffULL) continue;
                    const int waves = (int)ceil_div((u64)rt * ct * sb, 64);
                    const u64 groups = std::min<u64>({lds_max / b, (u64)(20 / waves), ceil_div(units, 256)});
                    const double busy = std::min(1.0, (double)(std::max<u64>(groups, 1) * waves) / 16.0);
                    const double fill = (double)(n0 * n2) / ((double)units * sb * ct * v) * ((double)(rt * ct * sb) / (64 * waves));
                    // narrow rows of a tile use part of a memory line, and
                    // each column of a thread shares its coefficients
                    const double line = std::min(1.0, 0.6 + 0.4 * cols * (double)elem_size / 64.0);
                    const double score = busy * fill * ((u64)cols == n2 ? 1.0 : line) * (v == 1 && n2 > 1 ? 0.8 : 1.0);
                    if (score <= best * 1.001) continue;
                    best = score;
                    sh.v = v;
                    sh.wrap = true;
                    a.rt = rt;
                    a.ct = ct;
                    a.sb = sb;
                    a.cb = cols;
                    a.pl = pitch;
                    a.rows = (int)n1;
                    a.nct = (int)ceil_div(n2, (u64)cols);
                    a.ns = ns > 0 ? ns : 64;  // staging and feet cost about 4 steps
                    a.units = (i64)units;
                    sh.threads = waves * 64;
                    sh.lds_bytes = b;
                    a.mcb = magic((u64)cols);
                }
            }
        }
        // long lines of many columns: segments of wider rows where only a few
        // columns of a whole line fit
        if (best >= 0.75 || (best > 0 && (n2 < 32 || whole_only))) {
            *out = sh;
            return true;
        }
        whole = best > 0;
        if (whole) *out = sh;
    }
    if (whole_only) return false;
    // segments
    sh.wrap = false;
    sh.v = n2 >= 3 ? 4 : (int)n2;
    a.ct = n2 > 4 ? 2 : 1;
    a.nct = (int)ceil_div(n2, (u64)a.ct * sh.v);
    a.cb = (int)ceil_div(n2, (u64)a.nct);
    a.rt = kSegment / a.ct;
    auto pitch = [&] { return plane_pitch(kTileLow + a.rt * kTileRows + kTileWin, a.cb); };
    while (a.rt > 64 && 2 * bytes(a.cb, pitch(), sh.v) > lds_max) a.rt -= 1;
    a.rows = a.rt * kTileRows;
    a.pl = pitch();
    a.mcb = magic((u64)a.cb);
    sh.threads = (int)ceil_div((u64)a.ct * a.rt, 64) * 64;
    sh.lds_bytes = bytes(a.cb, a.pl, sh.v);
    if ((u64)a.rows >= n1 || sh.lds_bytes > lds_max) return whole;
    const double s0 = p.minRealVx * p.dt * p.inv_dx;
    const double s1 = (p.minRealVx + (double)(n0 - 1) * p.dvx) * p.dt * p.inv_dx;
    a.hb_max = (int)std::max(0.0, std::floor(std::max(s0, s1) + 1e-6) + 3.0);
    a.ha_max = (int)std::max(0.0, 3.0 - std::floor(std::min(s0, s1) - 1e-6));
    const int hmax = std::max({7, a.hb_max, a.ha_max});  // of one slab (see tile_halo)
    if (ns <= 0) {
        // Steps per pass: staging, feet and stores cost about as much as kOver
        // steps, and the halo rows of all steps are computed at every step.
        const double over = sh.v == 1 ? 6.0 : 3.0;
        double best = 0;
        const u64 stride = std::max<u64>(1, n0 / 256);
        for (int k : {1, 2, 3, 4, 6, 8, 12, 16, 24, 32}) {
            if ((i64)k * hmax * 4 > (i64)a.rows * 3) break;
            double cost = 0;
            for (u64 i0 = 0; i0 < n0; i0 += stride) {
                int hb, ha;
                tile_halo(a.p, (i64)i0, a.hb_max, a.ha_max, hb, ha);
                cost += (over + k) / ((double)k * (a.rows - k * (hb + ha)));
            }
            if (ns <= 0 || cost < best) {
                best = cost;
                ns = k;
            }
        }
    }
    if (ns <= 0 || (i64)ns * hmax * 4 > (i64)a.rows * (whole ? 1 : 3)) return whole;
    a.ns = ns;
    a.hrows = ns * hmax;
    a.nseg = (int)ceil_div(n1, (u64)(a.rows - ns * hmax));
    a.units = (i64)n0 * a.nseg * a.nct;
    if ((u64)n0 * a.nseg * a.nct > 0x7fffffffULL) return whole;
    sh.halo_bytes = n0 * (u64)a.nseg * (u64)a.hrows * n2 * elem_size;
    *out = sh;
    return true;
}

bkma_status launch_tile(const TileShape &sh, bkma_dtype dt, bool fused, bool rnd, void *data, void *halo, int ns,
                        hipStream_t s) {
    if (ns < 1 || ns > sh.a.ns) return fail(BKMA_ERR_RUNTIME, "LINE_LDS tiles: steps per pass out of range");
    TileArgs a = sh.a;
    a.ns = ns;
    if (!sh.wrap) {  // fewer steps: smaller halos, longer segments (the snapshot keeps its row stride)
        const int h = a.hrows / sh.a.ns;
        a.nseg = (int)ceil_div((u64)a.p.n1, (u64)(a.rows - ns * h));
        a.units = a.p.n0 * a.nseg * a.nct;
    }
    if (dt == BKMA_F64) return launch_v<double, false, false>(sh, a, data, halo, s);
    if (rnd) return launch_v<float, true, true>(sh, a, data, halo, s);
    if (fused) return launch_v<float, true, false>(sh, a, data, halo, s);
    return launch_v<float, false, false>(sh, a, data, halo, s);
}

bkma_status launch_tile_group(const TileGroup &g, bkma_dtype dt, bool rnd, int ns, hipStream_t s) {
    if (ns < 1 || ns > g.ns) return fail(BKMA_ERR_RUNTIME, "LINE_LDS tiles: steps per pass out of range");
    if (dt == BKMA_F64) return launch_group_v<double, false, false>(g, ns, s);
    if (rnd) return launch_group_v<float, true, true>(g, ns, s);
    return launch_group_v<float, true, false>(g, ns, s);
}

}  // namespace bkma
