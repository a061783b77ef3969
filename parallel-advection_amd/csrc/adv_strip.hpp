// The LDS tiles of adv_tile.hpp with the steps themselves in registers: the
// strip form, for slabs whose shifts d = i1 - leftNode lie in
// [kStripDLo, kStripDHi].
//
// A wavefront holds a strip of 64 E consecutive rows of one column, E per
// lane, and advances it m steps on its own: the stencil's neighbours are the
// lane's own cells and those of the lanes around it, which arrive through DPP
// wavefront shifts (adv_shfl.hpp uses the same moves for lines that fill its
// work-group exactly).  A step spoils the rows next to the strip's ends, so
// neighbouring strips overlap: of 64 E rows, R are a strip's own and the
// others are the margins that m steps consume.  After m steps the strips
// exchange their rows through the LDS plane of the tile (two barriers).
// So LDS is read and written once per m steps instead of at every step, and
// lines of any length, columns and segments work as in the LDS form: WRAP
// tiles are whole lines, SEG tiles segments with halos.
//
// The window's first offset -d-2 is the same for all rows of a wavefront and a
// compile-time constant of the body that it selects.  A wavefront whose rows
// round to two shifts (slabs of shifts around an integer, such as the one at
// rest) runs a body that sums a row's own six cells out of a window of seven:
// 17 instructions per row instead of 11 (FP64).
#pragma once

#include "adv_shfl.hpp"
#include "adv_tile.hpp"

namespace bkma {

constexpr int kStripDLo = -5, kStripDHi = 6;
constexpr int kStripMaxThreads = 512;
constexpr int kStripSegE = 6;  // rows per lane of segments

// x of the lane H lanes down (H > 0) or up (H < 0) the wavefront; lanes
// without such a neighbour get 0 (they are margin).
template <int H> __device__ __forceinline__ double strip_shift(double x) {
    if constexpr (H == 0) return x;
    else if constexpr (H > 0) return strip_shift<H - 1>(dpp_rot_f64<kDppWaveShl1>(x));
    else return strip_shift<H + 1>(dpp_rot_f64<kDppWaveShr1>(x));
}

// g = one step of this lane's E cells f; windows start at offset DMIN.  MIXED:
// rows with their bit of `up` set (late rows) start one cell later; their
// coefficients are turned by one, the last one first.
template <bool FUSED, int E, int DMIN, bool MIXED>
__device__ __forceinline__ void strip_step(const double (&f)[E], double (&g)[E], const double (&c)[E][6], unsigned up) {
    constexpr int NW = E + 5 + (MIXED ? 1 : 0);
    double w[NW];
    static_for<0, NW>([&](auto tt) __attribute__((always_inline)) {
        constexpr int t = decltype(tt)::value;
        constexpr int o = DMIN + t;
        constexpr int hop = o >= 0 ? o / E : -((-o + E - 1) / E);
        w[t] = strip_shift<hop>(f[o - hop * E]);
    });
    if constexpr (MIXED) {
        // c[e][0] is the first tap of an early row and the last of a late one
#pragma unroll
        for (int e = 0; e < E; ++e) {
            const bool late = (up >> e) & 1;
            const double first = fma(c[e][0], w[e], 0.0);  // as tile_taps
            double acc = late ? 0.0 : first;
#pragma unroll
            for (int k = 1; k < 6; ++k) acc = FUSED ? fma(c[e][k], w[e + k], acc) : acc + c[e][k] * w[e + k];
            const double last = FUSED ? fma(c[e][0], w[e + 6], acc) : acc + c[e][0] * w[e + 6];
            g[e] = late ? last : acc;
        }
    } else {
        // a few rows tap by tap: FP64 results are ready after two issue slots
        constexpr int G = E % 3 == 0 ? 3 : 4;
#pragma unroll
        for (int e0 = 0; e0 < E; e0 += G) {
#pragma unroll
            for (int k = 0; k < 6; ++k) {
                double t[G];
#pragma unroll
                for (int e = 0; e < G; ++e) {
                    const double x = w[e0 + e + k];
                    if (k == 0) g[e0 + e] = fma(c[e0 + e][0], x, 0.0);
                    else if constexpr (FUSED) g[e0 + e] = fma(c[e0 + e][k], x, g[e0 + e]);
                    else t[e] = c[e0 + e][k] * x;
                }
                if constexpr (!FUSED) {
#pragma unroll
                    for (int e = 0; e < G; ++e)
                        if (k > 0) g[e0 + e] = g[e0 + e] + t[e];
                }
                __builtin_amdgcn_sched_barrier(0);
            }
        }
    }
}

template <bool FUSED, bool RND, int E, int DMIN, bool MIXED>
__device__ __forceinline__ void strip_steps(double (&f)[E], const double (&c)[E][6], unsigned up, int steps) {
    double g[E];
    auto round = [](double (&x)[E]) __attribute__((always_inline)) {
        if constexpr (RND) {
#pragma unroll
            for (int e = 0; e < E; ++e) x[e] = (double)(float)x[e];
        }
    };
    int s = 0;
    for (; s + 2 <= steps; s += 2) {
        strip_step<FUSED, E, DMIN, MIXED>(f, g, c, up);
        round(g);
        strip_step<FUSED, E, DMIN, MIXED>(g, f, c, up);
        round(f);
    }
    if (s < steps) {
        strip_step<FUSED, E, DMIN, MIXED>(f, g, c, up);
        round(g);
#pragma unroll
        for (int e = 0; e < E; ++e) f[e] = g[e];
    }
}

// The body of window start dmin (wave-uniform) in [D, DHI].
template <bool FUSED, bool RND, int E, bool MIXED, int D, int DHI>
__device__ __forceinline__ void strip_dispatch(int dmin, double (&f)[E], const double (&c)[E][6], unsigned up, int steps) {
    if constexpr (D <= DHI) {
        if (dmin == D) strip_steps<FUSED, RND, E, D, MIXED>(f, c, up, steps);
        else strip_dispatch<FUSED, RND, E, MIXED, D + 1, DHI>(dmin, f, c, up, steps);
    }
}

template <class T, bool FUSED, bool RND, int E, bool WRAP>
__device__ __forceinline__ void strip_unit(T *data, const T *__restrict__ halo, const TileArgs &a, i64 unit,
                                           double *__restrict__ lds) {
    constexpr int U = 8;
    const int n1 = (int)a.p.n1;
    const i64 n2 = a.p.n2;
    const int cb = a.cb, pl = a.pl, ns = a.ns, R = a.sr;
    const int slack = 64 * E - R;
    if constexpr (!WRAP) lds += slack;  // strips may start and end outside the buffer

    const i64 grp = unit / a.nct;
    const i64 col0 = (unit - grp * a.nct) * cb;
    const int cbw = (int)min((i64)cb, n2 - col0);
    i64 i0b;
    int nsl = 1, nrow, hbn = 0, r0 = 0, nr = 0, hb, m;
    const T *hsrc = nullptr;
    if constexpr (WRAP) {
        i0b = a.s0 + grp * a.sb;
        nsl = (int)min((i64)a.sb, a.s1 - i0b);
        nrow = nsl * n1;
        // steps between exchanges: the same for the tile's slabs (barriers)
        m = ns;
        for (int s = 0; s < nsl; ++s) {
            int b, f;
            tile_halo(a.p, i0b + s, a.hb_max, a.ha_max, b, f);
            m = min(m, slack / max(1, b + f));
        }
        m = max(1, m);
    } else {
        i0b = a.s0 + grp / a.nseg;
        const TileSeg s = tile_segment(a, i0b, (int)(grp % a.nseg));
        if (s.nr <= 0) return;  // uniform over the work-group
        hb = s.hb;
        hbn = ns * s.hb;
        r0 = s.r0;
        nr = s.nr;
        nrow = hbn + nr + ns * s.ha;
        hsrc = halo + grp * a.hrows * n2 + col0;
        m = max(1, slack / (s.hb + s.ha));
    }
    T *base = data + i0b * n1 * n2 + col0;
    tile_stage<T, U, WRAP>(a.apart ? halo + i0b * n1 * n2 + col0 : base, hsrc, lds, a, nrow, cbw, hbn, r0, nr);

    // ---- this wave's strip ----
    const int lane = (int)threadIdx.x & 63;
    const int wave = __builtin_amdgcn_readfirstlane((int)(threadIdx.x >> 6));
    const int pc = wave / a.strips, st = wave - pc * a.strips;
    const int sl = pc / a.ct, cc = pc - sl * a.ct;
    // wave-uniform; a segment's last strips may be beyond its rows
    const bool act = sl < nsl && (WRAP || st * R < nrow);
    if constexpr (WRAP) {
        int f;
        tile_halo(a.p, i0b + (act ? sl : 0), a.hb_max, a.ha_max, hb, f);
    }
    const int u0 = lane * E - m * hb;          // this lane's first row, from the strip's first own row
    const int own = WRAP ? min(R, n1 - st * R) : R;  // rows of the strip that are its own
    int r = st * R + u0;                       // tile row; WRAP: row of the line
    if constexpr (WRAP) {
        r %= n1;
        if (r < 0) r += n1;
    }
    double c[E][6];
    int d0 = 0;
    unsigned differ = 0;  // rows whose shift is not the wave's first
    const int half = n1 / 2;
    if (act) {
#pragma unroll
        for (int e = 0; e < E; ++e) {
            int lr = r + e;
            if constexpr (!WRAP) {
                lr += r0 - hbn;
                if (lr < 0) lr += n1;
            }
            if (lr >= n1) lr -= n1;
            lr = min(max(lr, 0), n1 - 1);  // rows far outside a segment's buffer: margin
            double d_prev1;
            int d = lr - tile_foot(a.p, (int)(i0b + sl), lr, d_prev1);
            adv_lag_basis(d_prev1, c[e]);
            if (d > half) d -= n1;
            if (d < -half) d += n1;
            if (e == 0) d0 = __builtin_amdgcn_readfirstlane(d);
            differ |= (unsigned)(d != d0) << e | (unsigned)(d > d0) << (16 + e);
            __builtin_amdgcn_sched_barrier(0);  // one row's temporaries at a time
        }
    }
    // two adjacent shifts at most: the window starts at the larger one's, the
    // rows of the smaller start one cell later
    const bool mixed = __any(differ != 0);
    const int dmax = __any((differ >> 16) != 0) ? d0 + 1 : d0;
    const unsigned up = dmax > d0 ? ~(differ >> 16) : differ & 0xffffu;
    if (mixed) {
#pragma unroll
        for (int e = 0; e < E; ++e) {
            const bool late = (up >> e) & 1;
            const double c5 = c[e][5];
#pragma unroll
            for (int k = 5; k > 0; --k) c[e][k] = late ? c[e][k - 1] : c[e][k];
            c[e][0] = late ? c5 : c[e][0];
        }
    }
    const int dmin = min(max(-dmax - 2, -kStripDHi - 2), -kStripDLo - 2);
    __syncthreads();

    // ---- blocks of m steps ----
    const int nv = (cbw + a.ct - 1) / a.ct;  // columns per wave in this tile (uniform)
    for (int s = 0; s < ns; s += m) {
        const int steps = min(m, ns - s);
        double *w = lds + (sl * cb + cc) * pl;
        int col = act ? cc : cbw;
#pragma unroll 1
        for (int v = 0; v < nv; ++v) {
            const bool on = col < cbw;
            double f[E];
            if (on) {
#pragma unroll
                for (int e = 0; e < E; ++e) f[e] = w[r + e];
                if (!mixed) strip_dispatch<FUSED, RND, E, false, -kStripDHi - 2, -kStripDLo - 2>(dmin, f, c, up, steps);
                else strip_dispatch<FUSED, RND, E, true, -kStripDHi - 2, -kStripDLo - 2>(dmin, f, c, up, steps);
            }
            __syncthreads();
            if (on) {
                double *dst = w + st * R + u0;
                if (u0 >= 0 && u0 + E <= own) {
#pragma unroll
                    for (int e = 0; e < E; ++e) dst[e] = f[e];
                } else {
#pragma unroll
                    for (int e = 0; e < E; ++e)
                        if (u0 + e >= 0 && u0 + e < own) dst[e] = f[e];
                }
                if constexpr (WRAP) {
                    if (st * R + u0 < kTileGhost) {
#pragma unroll
                        for (int e = 0; e < E; ++e)
                            if (u0 + e >= 0 && u0 + e < own && st * R + u0 + e < kTileGhost) dst[n1 + e] = f[e];
                    }
                }
            }
            w += a.ct * pl;
            col += a.ct;
        }
        if (nv == 1) __syncthreads();
    }
    if (nv > 1) __syncthreads();
    const int nout = WRAP ? nrow : nr;
    tile_store<T, U, WRAP>(base, lds, a, nout, cbw, hbn, r0);
}

}  // namespace bkma
