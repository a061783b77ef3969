// Kernels, launch shapes and launchers of the LDS tile form with register
// coefficients (adv_tile.hpp).
#include <algorithm>
#include <cmath>

#include "adv_strip.hpp"

namespace bkma {

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

template <class T, bool FUSED, bool RND, int V, bool WRAP>
bkma_status launch(const TileShape &sh, const TileArgs &a, void *data, void *halo, hipStream_t s) {
    static std::atomic<unsigned> done{0};
    auto k = adv_tile_kernel<T, FUSED, RND, V, WRAP>;
    BKMA_TRY(allow_lds(k, done));
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
    if (sh.v == 1) return launch<T, FUSED, RND, 1, false>(sh, a, data, halo, s);
    if (sh.v == 2) return launch<T, FUSED, RND, 2, false>(sh, a, data, halo, s);
    return launch<T, FUSED, RND, 4, false>(sh, a, data, halo, s);
}

template <class T, bool FUSED, bool RND, int V, bool WRAP>
bkma_status launch_group(const TileGroup &g, int ns, hipStream_t s) {
    static std::atomic<unsigned> done{0};
    auto k = adv_tile_group_kernel<T, FUSED, RND, V, WRAP>;
    BKMA_TRY(allow_lds(k, done));
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

namespace {

// Quotients of tile indexes by the columns of a row, and whether its rows can
// be moved 16 bytes at a time.
void set_columns(TileArgs &a, u64 cols, u64 elem_size) {
    const u64 w = 16 / elem_size;
    a.mcb = magic(cols);
    a.wide = cols % w == 0 && (u64)a.p.n2 % w == 0;
    a.mcw = a.wide ? magic(cols / w) : a.mcb;
}

// Largest halo rows per step of the slabs [a.s0, a.s1) on either side, and
// (returned) on both sides of one of them: 5 rows, 6 with two shifts, more
// where the shift leaves the stencil on one side.
int halo_bounds(TileArgs &a) {
    double lo0, hi0, lo1, hi1;
    tile_shifts(a.p, a.s0, lo0, hi0);
    tile_shifts(a.p, a.s1 - 1, lo1, hi1);
    a.hb_max = (int)std::max(0.0, std::max(hi0, hi1) + 2.0);
    a.ha_max = (int)std::max(0.0, 3.0 - std::min(lo0, lo1));
    return std::max({6, a.hb_max, a.ha_max});
}

// Steps per pass of a segment tile of `rows` rows: staging, feet and stores
// cost about as much as `over` steps, and the halo rows of all steps are
// computed at every step.
int segment_steps(const TileArgs &a, int rows, int hmax, double over) {
    int ns = 0;
    double best = 0;
    const i64 stride = std::max<i64>(1, (a.s1 - a.s0) / 256);
    for (int k : {1, 2, 3, 4, 6, 8, 12, 16, 24, 32, 64}) {
        if ((i64)k * hmax * 4 > (i64)rows * 3) break;
        double cost = 0;
        for (i64 i0 = a.s0; i0 < a.s1; i0 += stride) {
            int hb, ha;
            tile_halo(a.p, i0, a.hb_max, a.ha_max, hb, ha);
            cost += (over + k) / ((double)k * (rows - k * (hb + ha)));
        }
        if (ns == 0 || cost < best) {
            best = cost;
            ns = k;
        }
    }
    return ns;
}

// Segments of a.rows buffer rows and passes of ns steps; false where they do
// not fit.
bool set_segments(TileShape &sh, int ns, int hmax, u64 elem_size) {
    TileArgs &a = sh.a;
    if (ns <= 0 || (i64)ns * hmax * 4 > (i64)a.rows * 3) return false;
    a.ns = ns;
    a.hrows = ns * hmax;
    a.nseg = (int)ceil_div((u64)a.p.n1, (u64)(a.rows - a.hrows));
    a.units = (a.s1 - a.s0) * a.nseg * a.nct;
    if ((u64)a.units > 0x7fffffffULL || (i64)a.nseg * a.nct > tile_launch_units(sh.threads)) return false;
    sh.halo_bytes = (u64)(a.s1 - a.s0) * (u64)a.nseg * (u64)a.hrows * (u64)a.p.n2 * elem_size;
    return true;
}

}  // namespace

bool tile_shape(const bkma_adv_params &p, u64 s0, u64 s1, u64 elem_size, int ns, u64 lds_max, TileShape *out,
                bool whole_only) {
    if (p.n1 < 16 || s1 <= s0 || p.n2 == 0) return false;
    // Threads per work-group.  Whole lines: work-groups of four wavefronts,
    // five to a CU, keep the LDS and the VALU busy at different times
    // ([2048][1024][64] FP64, 20 steps: 1436 Gcell/s with 205 threads, 1290
    // with 410).  Segments: longer ones have fewer halo rows.
    constexpr int kWhole = 256, kSegment = 512;
    const u64 n0 = s1 - s0, n1 = p.n1, n2 = p.n2;
    TileShape sh;
    TileArgs &a = sh.a;
    a.p = make_adv_dev(p);
    a.s0 = (i64)s0;
    a.s1 = (i64)s1;
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
                    a.ns = ns > 0 ? ns : kTileMaxSteps;  // staging and feet cost about 4 steps
                    a.units = (i64)units;
                    sh.threads = waves * 64;
                    sh.lds_bytes = b;
                    set_columns(a, (u64)cols, elem_size);
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
    set_columns(a, (u64)a.cb, elem_size);
    sh.threads = (int)ceil_div((u64)a.ct * a.rt, 64) * 64;
    sh.lds_bytes = bytes(a.cb, a.pl, sh.v);
    if ((u64)a.rows >= n1 || sh.lds_bytes > lds_max) return whole;
    const int hmax = halo_bounds(a);
    if (ns <= 0) ns = segment_steps(a, a.rows, hmax, sh.v == 1 ? 6.0 : 3.0);
    if (whole && (i64)ns * hmax * 4 > (i64)a.rows) return true;  // *out is the whole-line tile
    if (!set_segments(sh, ns, hmax, elem_size)) return whole;
    *out = sh;
    return true;
}

bool strip_shape(const bkma_adv_params &p, u64 s0, u64 s1, u64 elem_size, int ns, u64 lds_max, TileShape *out) {
    if (p.n1 < 16 || s1 <= s0 || p.n2 == 0) return false;
    const u64 n0 = s1 - s0, n1 = p.n1, n2 = p.n2;
    TileShape sh;
    TileArgs &a = sh.a;
    a.p = make_adv_dev(p);
    a.s0 = (i64)s0;
    a.s1 = (i64)s1;
    a.sb = 1;
    a.nseg = 1;
    a.mn1 = magic(n1);
    const int hmax = halo_bounds(a);
    // What a shape is worth: the part of the lanes' rows that are rows of the
    // line, and the time lost to the exchange after m steps (a step or two,
    // eight where no other work-group runs beside it), the two DPP moves per
    // neighbour cell (10 per lane and step), the feet (shared by the `cols / ct`
    // columns of a wave), SIMDs with one or two wavefronts (latency),
    // work-groups too few to be in different phases, wavefronts that the SIMDs
    // do not share evenly, idle CUs of the last round, narrow rows.
    auto worth = [&](int e, int strips, double rows, int m, int cols, int ct, int sb, u64 units, u64 lds) {
        const double taps = elem_size == 8 ? 11.0 : 6.0;
        const int waves = sb * strips * ct, resident = e == 8 ? 12 : e == 6 ? 16 : 20;
        const u64 groups = std::max<u64>(std::min<u64>({lds_max / lds, (u64)(resident / waves), ceil_div(units, 256)}), 1);
        const double per_simd = (double)groups * waves / 4.0, depth = std::ceil(per_simd);
        const double busy = (depth <= 1 ? 0.6 : depth <= 2 ? 0.74 : depth <= 3 ? 0.86 : depth <= 4 ? 0.95 : 1.0) * per_simd / depth;
        const double apart = 1.0 - 0.25 / (double)groups - 0.01 * (waves - 1) - (groups <= 2 && waves % 4 ? 0.15 : 0.0);
        const double fill = (double)n2 / ((double)ceil_div(n2, (u64)cols) * ct * ceil_div((u64)cols, (u64)ct));
        const double line = (u64)cols == n2 ? 1.0 : std::min(1.0, 0.9 + 0.1 * cols * (double)elem_size / 32.0);
        const double cus = (double)units / (256.0 * ceil_div(units, 256));
        const bool wide = cols % (16 / (int)elem_size) == 0 && n2 % (16 / elem_size) == 0;
        return rows * m / (m + 0.5 + 8.0 / (double)groups) * taps / (taps + 10.0 / e) * busy * apart * fill * line * cus *
               (wide || n2 == 1 ? 1.0 : 0.93) / (1.0 + 0.2 * ct / cols);
    };
    double best = 0;
    // Segments: four strips of 384 rows with four steps between exchanges, up
    // to four columns one after the other (best or within 3% of it on five
    // problems, over 2 to 8 strips of 256 to 512 rows, 2 to 12 steps, 1 to 8
    // columns).  The rows of all steps' halos are computed too.
    const int sr = 64 * kStripSegE - 4 * hmax;
    if ((u64)(4 * sr) < n1) {
        sh.wrap = false;
        sh.e = kStripSegE;
        a.ct = 1;
        a.strips = 4;
        a.nct = (int)ceil_div(n2, (u64)4);
        a.cb = (int)ceil_div(n2, (u64)a.nct);
        a.sr = sr;
        a.rows = 4 * sr;
        a.pl = plane_pitch(a.rows + 2 * 4 * hmax, a.cb);
        set_columns(a, (u64)a.cb, elem_size);
        sh.threads = 64 * a.strips;
        sh.lds_bytes = ((u64)a.cb * a.pl + 4 * (u64)hmax) * 8;
        if (sh.lds_bytes <= lds_max && set_segments(sh, ns > 0 ? ns : segment_steps(a, a.rows, hmax, 16.0), hmax, elem_size)) {
            const u64 len = ceil_div(n1, (u64)a.nseg) + (u64)a.hrows;
            const double rows = (double)n1 / ((double)a.nseg * ceil_div(len, (u64)sr) * 64 * kStripSegE);
            best = 0.95 * worth(sh.e, 4, rows, 4, a.cb, 1, 1, (u64)a.units, sh.lds_bytes);  // the snapshot
            *out = sh;
        }
    }
    // Whole lines.  Over all shapes of eleven problems of 64 to 3000 rows the
    // choice is within 6% of the fastest, save [1000][300][1] (24 us; two
    // 256-row strips of two slabs 17).  Segments win from about 2500 rows on: at
    // 20 steps and [n][n1][8], FP64, whole 0.55 ms and segments 0.61 with 2000
    // rows, 0.80 and 0.52 with 2500, 0.65 and 0.55 with 3500.
    sh.wrap = true;
    sh.halo_bytes = 0;
    a.nseg = 1;
    a.hrows = 0;
    for (int e : {8, 6, 4}) {
        const int reach = 64 * e;
        if (reach <= hmax) continue;
        const int least = (int)std::min<u64>(ceil_div(n1, (u64)(reach - hmax)), 99);
        for (int strips = least; strips <= std::min(least + 2, kStripMaxThreads / 64); ++strips) {
            const int own = (int)ceil_div(n1, (u64)strips);
            const int m = (reach - own) / hmax;
            if (m < 1) continue;
            if (strips > least && (reach - (int)ceil_div(n1, (u64)least)) / hmax >= 16) break;  // few exchanges already
            for (int ct = 1; strips * ct * 64 <= kStripMaxThreads && (u64)ct <= n2; ++ct) {
                for (int v = 1; v <= 4 && (u64)(v - 1) * ct < n2; ++v) {
                    const u64 nct = ceil_div(n2, (u64)ct * v);
                    const int cols = (int)ceil_div(n2, nct);
                    const int pitch = plane_pitch((int)n1 + kTileGhost, cols);
                    for (int sb = 1; sb * strips * ct * 64 <= kStripMaxThreads && (u64)sb <= n0 && (sb == 1 || (u64)cols == n2); ++sb) {
                        const u64 b = (u64)sb * cols * pitch * 8;
                        const u64 units = ceil_div(n0, (u64)sb) * nct;
                        if (b > lds_max || units > 0x7fffffffULL) continue;
                        const double score = worth(e, strips, (double)n1 / ((double)strips * reach), m, cols, ct, sb, units, b);
                        if (score <= best * 1.001) continue;
                        best = score;
                        sh.e = e;
                        a.strips = strips;
                        a.sr = own;
                        a.ct = ct;
                        a.sb = sb;
                        a.cb = cols;
                        a.nct = (int)nct;
                        a.pl = pitch;
                        a.rows = (int)n1;
                        a.ns = ns > 0 ? ns : kTileMaxSteps;
                        a.units = (i64)units;
                        set_columns(a, (u64)cols, elem_size);
                        sh.threads = 64 * sb * strips * ct;
                        sh.lds_bytes = b;
                        *out = sh;
                    }
                }
            }
        }
    }
    return best > 0;
}

std::vector<TileShape> tile_parts(const bkma_adv_params &p, u64 elem_size, int ns, u64 lds_max, bool strips) {
    std::vector<TileShape> parts;
    TileShape all;
    if (!tile_covers(make_adv_dev(p)) || !tile_shape(p, 0, p.n0, elem_size, ns, lds_max, &all)) return parts;
    // Slabs [lo, hi) whose shifts the strips cover (monotone in the slab).
    const AdvDev d = make_adv_dev(p);
    auto covered = [&](u64 i0) {
        double dlo, dhi;
        tile_shifts(d, (i64)i0, dlo, dhi);
        return dlo >= (double)kStripDLo && dhi <= (double)kStripDHi;
    };
    // the slab nearest to s = 0, and from it the ends by bisection
    const double step = d.dvx * d.dt * d.inv_dx, first = d.minRealVx * d.dt * d.inv_dx;
    const double at = step != 0.0 ? -first / step : 0.0;
    const u64 mid = at > 0.0 ? (at < (double)(p.n0 - 1) ? (u64)at : p.n0 - 1) : 0;
    u64 lo = mid, hi = mid;
    if (covered(mid)) {
        u64 a = 0, b = mid;  // first covered slab
        while (a < b) {
            const u64 c = (a + b) / 2;
            if (covered(c)) b = c;
            else a = c + 1;
        }
        lo = a;
        a = mid;
        b = p.n0;  // first slab past them
        while (a < b) {
            const u64 c = (a + b) / 2;
            if (covered(c)) a = c + 1;
            else b = c;
        }
        hi = a;
    }
    TileShape strip;
    // a split costs a launch and its tail: it has to cover a good part
    if (!strips || (hi - lo) * 4 < p.n0 || !strip_shape(p, lo, hi, elem_size, ns > 0 || hi - lo == p.n0 ? ns : all.a.ns, lds_max, &strip)) {
        parts.push_back(all);
        return parts;
    }
    for (int side = 0; side < 2; ++side) {
        const u64 b = side ? hi : 0, e = side ? p.n0 : lo;
        TileShape t;
        if (b == e) continue;
        if (!tile_shape(p, b, e, elem_size, strip.a.ns, lds_max, &t)) {
            parts.assign(1, all);
            return parts;
        }
        parts.push_back(t);
    }
    parts.insert(parts.begin(), strip);
    return parts;
}

namespace {

// One pass over the slabs [a.s0, a.s1).
bkma_status launch_slabs(const TileShape &sh, const TileArgs &a, bkma_dtype dt, bool fused, bool rnd, void *data,
                         void *halo, hipStream_t s, void *from) {
    if (!sh.wrap && !from) {
        const unsigned groups = (unsigned)((a.s1 - a.s0) * a.nseg);
        const unsigned nt = (i64)a.hrows * a.p.n2 >= 512 ? 256 : 64;
        if (dt == BKMA_F64)
            hipLaunchKernelGGL(tile_snapshot_kernel<double>, dim3(groups), dim3(nt), 0, s, (const double *)data, (double *)halo, a);
        else
            hipLaunchKernelGGL(tile_snapshot_kernel<float>, dim3(groups), dim3(nt), 0, s, (const float *)data, (float *)halo, a);
        BKMA_TRY(check_launch("tile_snapshot_kernel"));
    }
    if (sh.e) {
        if (dt == BKMA_F64) return launch_strip_f64(sh, a, data, halo, s);
        if (rnd) return launch_strip_f32_round(sh, a, data, halo, s);
        if (fused) return launch_strip_f32(sh, a, data, halo, s);
        return fail(BKMA_ERR_RUNTIME, "LINE_LDS strips: FP32 sums are fused");
    }
    if (dt == BKMA_F64) return launch_v<double, false, false>(sh, a, data, halo, s);
    if (rnd) return launch_v<float, true, true>(sh, a, data, halo, s);
    if (fused) return launch_v<float, true, false>(sh, a, data, halo, s);
    return launch_v<float, false, false>(sh, a, data, halo, s);
}

}  // namespace

bkma_status launch_tile(const TileShape &sh, bkma_dtype dt, bool fused, bool rnd, void *data, void *halo, int ns,
                        hipStream_t s, void *from) {
    if (ns < 1 || ns > sh.a.ns) return fail(BKMA_ERR_RUNTIME, "LINE_LDS tiles: steps per pass out of range");
    TileArgs a = sh.a;
    a.ns = ns;
    if ((uintptr_t)data % 16 != 0) a.wide = 0;
    if (from) {
        a.apart = 1;
        halo = from;
    }
    if (!sh.wrap) {  // fewer steps: smaller halos, longer segments (the snapshot keeps its row stride)
        const int h = a.hrows / sh.a.ns;
        a.nseg = (int)ceil_div((u64)a.p.n1, (u64)(a.rows - ns * h));
    }
    // HIP launches have fewer than 2^32 threads: slabs in several launches where
    // they need more ([2^24][1000][1]: one work-group of 256 per slab)
    const i64 per = tile_slabs_per_launch(sh, a.nseg);
    for (i64 s0 = sh.a.s0; s0 < sh.a.s1; s0 += per) {
        a.s0 = s0;
        a.s1 = std::min(s0 + per, sh.a.s1);
        a.units = sh.wrap ? (i64)ceil_div((u64)(a.s1 - a.s0), (u64)a.sb) * a.nct : (a.s1 - a.s0) * a.nseg * a.nct;
        BKMA_TRY(launch_slabs(sh, a, dt, fused, rnd, data, halo, s, from));
    }
    return BKMA_OK;
}

bkma_status launch_tile_group(const TileGroup &g, bkma_dtype dt, bool rnd, int ns, hipStream_t s) {
    if (ns < 1 || ns > g.ns) return fail(BKMA_ERR_RUNTIME, "LINE_LDS tiles: steps per pass out of range");
    if (!g.wrap) {
        const auto k = dt == BKMA_F64 ? tile_group_snapshot_kernel<double> : tile_group_snapshot_kernel<float>;
        hipLaunchKernelGGL(k, dim3((unsigned)g.halo_units), dim3(256), 0, s, (const TileProblem *)g.table, g.count, ns);
        BKMA_TRY(check_launch("tile_group_snapshot_kernel"));
    }
    if (g.e) {
        if (dt == BKMA_F64) return launch_strip_group_f64(g, ns, s);
        return rnd ? launch_strip_group_f32_round(g, ns, s) : launch_strip_group_f32(g, ns, s);
    }
    if (dt == BKMA_F64) return launch_group_v<double, false, false>(g, ns, s);
    if (rnd) return launch_group_v<float, true, true>(g, ns, s);
    return launch_group_v<float, true, false>(g, ns, s);
}

}  // namespace bkma
