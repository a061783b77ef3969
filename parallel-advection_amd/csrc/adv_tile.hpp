// Advection steps fused in LDS with the coefficients in registers (the
// register form of strategy LINE_LDS, see bkma_tuned.hip).
//
// A work-group owns a tile: kTileRows consecutive rows per thread of one
// column of one slab, RT threads along the rows, CT threads times V columns
// across, SB slabs.  The tile's values live in LDS as FP64, one plane of
// rows per (slab, column); a thread computes the foot and the six
// coefficients of its rows once per pass and keeps them in registers for all
// the steps of the pass, since they depend on (i0, i1) only.  A step reads the
// kTileRows + 5 rows around a thread's shifted position (consecutive LDS
// addresses, immediate offsets) and writes its kTileRows results back, so a
// cell costs 3 LDS accesses and 6 multiply-adds per step; the foot arithmetic
// (about 55 FP64 instructions per row) and HBM are paid once per pass.
//  - WRAP tiles hold whole lines.  The first rows are repeated after the last
//    one, so a window never wraps inside.  A pass may fuse any number of
//    steps.
//  - SEG tiles hold a segment of a longer line and the halo rows that the
//    pass's steps reach (per slab: 5 rows per step, |s| + 3 where the shift
//    leaves the stencil on one side), every row of the
//    buffer is computed at every step and the rows next to the ends, which
//    read outside the buffer, are discarded as the halo shrinks.  Rows that
//    other work-groups overwrite in the same pass come from a snapshot.
// Five rows per thread: the LDS row stride of neighbouring threads is then 5
// doubles, which spreads 32 lanes over all 64 banks, and the coefficients take
// 60 VGPRs, which leaves 4 wavefronts per SIMD.
//
// What bounds it: at 20 steps on [512][1024][512] the VALU is 58% and the LDS
// 55% busy (FP32 storage 45% and 64%), with two work-groups per CU whose
// barriers alternate the two.  Measured (steps kernel before -> this one):
//   [300][1000][100]    FP64, 20 steps   2.93 -> 0.45 ms (column pair before)
//   [4096][10000][1]    FP64, 20 steps  11.68 -> 0.67 ms
//   [256][262144][4]    FP32, 20 steps  12.93 -> 5.7 ms (halo rows are 28% of
//                       a tile there, the shifts reach 262 cells; 6.4 ms with
//                       a snapshot in every pass)
//   [512][1024][512]    20 steps        1440 Gcell/s FP64, 1620 FP32
// Slabs with shifts of a few cells take the strips of adv_strip.hpp instead.
// Rows of one thread that round to different shifts (a slab whose shift is an
// integer up to rounding) take a form that reads every row's own six taps.
//
// Arithmetic: FP64 with the reference's separately rounded products and sums
// (FUSED = false), or fused (FP32 storage in the plans).  RND rounds the
// values to FP32 after every step: a pass then equals as many passes of one
// step each.
#pragma once

#include <algorithm>
#include <atomic>
#include <climits>
#include <cmath>
#include <vector>

#include "common.hpp"

namespace bkma {

constexpr int kTileRows = 5;               // rows per thread
constexpr int kTileWin = kTileRows + 5;    // rows a thread's step reads
constexpr int kStripForm = 6;  // bkma_tuned_config::prefetch of the strip form (kTileRows: of the LDS form)
constexpr int kTileGhost = 2 * kTileRows;  // rows repeated after a whole line
constexpr int kTileLow = kTileRows;        // SEG: rows a thread's window may start before the buffer
constexpr int kTileThreads = 1024;         // largest work-group
constexpr int kTileMaxSteps = 256;         // steps per pass

struct TileArgs {
    AdvDev p;
    int rt, ct, cb, sb;  // row threads per plane, column threads, columns and slabs per tile
    int nct;             // column tiles per slab
    int rows;            // SEG: rows of the buffer (rt * kTileRows)
    int pl;              // plane pitch in doubles
    int ns;              // steps in this pass
    int nseg;            // SEG: work-groups per (slab, column tile); a slab uses as many as its halos need
    int hb_max, ha_max;  // SEG: largest halo rows per step before and after a segment
    int hrows;           // SEG: snapshot rows per (slab, segment)
    unsigned mcb, mn1;   // ceil(2^32 / cb) (cb > 1), ceil(2^32 / n1): quotients of tile indexes (below 2^16)
    unsigned mcw;        // ceil(2^32 / (cb / W)), W elements of 16 bytes
    int wide;            // staged and stored 16 bytes at a time: columns and addresses allow it
    int strips, sr;      // strip form: wavefronts per plane, rows of a strip that are its own
    int apart;           // rows come from another array (the kernels' `halo`), nothing is overwritten
    i64 s0, s1;          // the launch's slabs
    i64 units;
};

// Smallest and largest shift of slab i0: d = i1 - leftNode is ceil(s),
// s = v dt / dx, up to the rounding of the foot (some ulps of the coordinates).
__host__ __device__ __forceinline__ void tile_shifts(const AdvDev &p, i64 i0, double &dlo, double &dhi) {
    const double s = (p.minRealVx + (double)(int)i0 * p.dvx) * p.dt * p.inv_dx;
    const double e = 1e-6 + 1e-15 * (fabs(p.minRealX) + 2.0 * p.realWidthX) * p.inv_dx;
    dlo = ceil(s - e);
    dhi = ceil(s + e);
}

// Whether tile_shifts holds for every slab of the problem, as all tiles take
// for granted: a regular periodic grid (the derived fields agree to a small part
// of the 1e-6 above, added up over a line), coordinates that resolve the cells,
// so that a slab's rows take at most two adjacent shifts, and shifts below half
// a line.  The executors' own kernels, and the others, evaluate any foot.
inline bool tile_covers(const AdvDev &p) {
    const double n1 = (double)p.n1, v1 = p.minRealVx + (double)(p.n0 - 1) * p.dvx;
    const double s = std::fabs(p.dt * p.inv_dx) * std::max(std::fabs(p.minRealVx), std::fabs(v1));
    const double apart = n1 * (std::fabs(p.dx * p.inv_dx - 1.0) + std::fabs(p.dx * n1 / p.realWidthX - 1.0));
    const double round = 1e-15 * (std::fabs(p.minRealX) + 2.0 * p.realWidthX) * p.inv_dx;
    return p.realWidthX > 0 && std::isfinite(p.realWidthX) && p.n0 <= INT_MAX && p.n1 <= INT_MAX && apart <= 5e-7 &&
           round <= 0.25 && s + 4.0 < n1 / 2.0;  // NaN is false
}

// Halo rows per step of slab i0 before and after a segment (the stencil of
// row i1 reads rows i1-d-2 .. i1-d+3).
__host__ __device__ __forceinline__ void tile_halo(const AdvDev &p, i64 i0, int hb_max, int ha_max, int &hb, int &ha) {
    double dlo, dhi;
    tile_shifts(p, i0, dlo, dhi);
    const double b = dhi + 2.0 > 0.0 ? dhi + 2.0 : 0.0, a = 3.0 - dlo > 0.0 ? 3.0 - dlo : 0.0;
    hb = b < (double)hb_max ? (int)b : hb_max;
    ha = a < (double)ha_max ? (int)a : ha_max;
}

// Segment `seg` of slab i0: rows [r0, r0 + nr) with ns*hb and ns*ha halo rows.
struct TileSeg {
    int hb, ha, r0, nr;
};
__device__ __forceinline__ TileSeg tile_segment(const TileArgs &a, i64 i0, int seg) {
    TileSeg s;
    tile_halo(a.p, i0, a.hb_max, a.ha_max, s.hb, s.ha);
    const int n1 = (int)a.p.n1;
    const int cap = a.rows - a.ns * (s.hb + s.ha);
    const int cnt = (n1 + cap - 1) / cap;
    const int len = (n1 + cnt - 1) / cnt;
    s.r0 = seg * len;
    s.nr = min(len, n1 - s.r0);  // <= 0: the slab needs fewer segments
    return s;
}

// Old rows around every segment: ns*hb rows before it, then ns*ha after it
// (periodic), hrows rows of n2 columns per (slab, segment).
template <class T>
__device__ __forceinline__ void tile_snapshot_unit(const T *__restrict__ data, T *__restrict__ halo, const TileArgs &a,
                                                   i64 unit) {
    const i64 i0 = a.s0 + unit / a.nseg;
    const TileSeg s = tile_segment(a, i0, (int)(unit % a.nseg));
    if (s.nr <= 0) return;
    const i64 n2 = a.p.n2, line = a.p.n1 * n2;
    const T *slab = data + i0 * line;
    T *dst = halo + unit * a.hrows * n2;
    const i64 before = (i64)a.ns * s.hb * n2, total = before + (i64)a.ns * s.ha * n2;
    const i64 b0 = (i64)s.r0 * n2 - before, a0 = (i64)(s.r0 + s.nr) * n2 - before;
    for (i64 e = threadIdx.x; e < total; e += blockDim.x) {
        i64 src = e + (e < before ? b0 : a0);
        if (src < 0) src += line;
        if (src >= line) src -= line;
        dst[e] = slab[src];
    }
}

// adv_foot for |v*dt| below half the width (every tile's caller checks it):
// the argument of the periodic remainder lies in [0, 3W), where a - W and
// a - 2W are exact, so no library fmod is needed.
__device__ __forceinline__ int tile_foot(const AdvDev &p, int i0, int i1, double &d_prev1) {
    const double x = adv_coord(i1, p.minRealX, p.dx);
    const double vx = adv_coord(i0, p.minRealVx, p.dvx);
    const double displx = p.dt * vx;
    const double a = p.realWidthX + x - displx - p.minRealX, w2 = 2.0 * p.realWidthX;
    const double xFoot = p.minRealX + (a - (a >= w2 ? w2 : a >= p.realWidthX ? p.realWidthX : 0.0));
    const int leftNode = (int)floor((xFoot - p.minRealX) * p.inv_dx);
    d_prev1 = 2 + p.inv_dx * (xFoot - adv_coord(leftNode, p.minRealX, p.dx));
    return leftNode;
}

// W elements of T in one access of 16 bytes (W = 1: one element).
template <class T, int W> struct alignas(W == 1 ? alignof(T) : 16) TilePack {
    T v[W];
};

// Stages the tile's rows as FP64, about U elements in flight per thread.
// WRAP: whole lines of all slabs of the tile, their first kTileGhost rows also
// after the last; SEG: hbn halo rows, nr rows from line row r0 on, the other
// halo rows.  W > 1: rows of 16-byte accesses, a.cb and n2 multiples of W.
// Index arithmetic is most of what an element costs here (strips, [512][1024][512],
// one step: FP32 0.98 ms with W = 1, 0.88 with W = 4; FP64 1.29 and 1.13 ms).
template <class T, int U, int W, bool WRAP>
__device__ __forceinline__ void tile_stage_w(const T *base, const T *__restrict__ hsrc, double *__restrict__ lds,
                                             const TileArgs &a, int nrow, int cbw, int hbn, int r0, int nr) {
    constexpr int UW = W == 1 ? U : U / 2;  // accesses in flight
    const int n1 = (int)a.p.n1, tid = (int)threadIdx.x, nthr = (int)blockDim.x, cb = a.cb;
    const unsigned cq = (unsigned)(cb / W), mq = W == 1 ? a.mcb : a.mcw;
    const i64 n2 = a.p.n2;
    const int total = nrow * (int)cq;
#pragma unroll 1
    for (int q0 = tid; q0 < total; q0 += UW * nthr) {
        TilePack<T, W> ld[UW];
#pragma unroll
        for (int i = 0; i < UW; ++i) {
            const unsigned q = (unsigned)(q0 + i * nthr);
            const unsigned row = cq == 1 ? q : __umulhi(q, mq);
            const unsigned col = (q - row * cq) * W;
#pragma unroll
            for (int k = 0; k < W; ++k) ld[i].v[k] = (T)0;
            if ((int)row < nrow && (int)col < cbw) {
                const T *src;
                if constexpr (WRAP) {
                    src = base + (i64)row * n2;
                } else if (a.apart) {
                    int lr = r0 - hbn + (int)row;
                    lr += lr < 0 ? n1 : lr >= n1 ? -n1 : 0;
                    src = base + (i64)lr * n2;
                } else {
                    const int b = (int)row - hbn;
                    src = b >= 0 && b < nr ? base + (i64)(r0 + b) * n2 : hsrc + (i64)(b < 0 ? (int)row : (int)row - nr) * n2;
                }
                ld[i] = *reinterpret_cast<const TilePack<T, W> *>(src + col);
            }
        }
#pragma unroll
        for (int i = 0; i < UW; ++i) {
            const unsigned q = (unsigned)(q0 + i * nthr);
            unsigned row = cq == 1 ? q : __umulhi(q, mq);
            const unsigned col = (q - row * cq) * W;
            if ((int)row < nrow && (int)col < cbw) {
                unsigned s = 0;
                if constexpr (WRAP) {
                    s = __umulhi(row, a.mn1);
                    row -= s * (unsigned)n1;
                }
                double *dst = lds + (int)(s * (unsigned)cb + col) * a.pl + (int)row;
#pragma unroll
                for (int k = 0; k < W; ++k) dst[k * a.pl] = (double)ld[i].v[k];
                if constexpr (WRAP) {
                    if ((int)row < kTileGhost) {
#pragma unroll
                        for (int k = 0; k < W; ++k) dst[k * a.pl + n1] = (double)ld[i].v[k];
                    }
                }
            }
        }
    }
}

// The tile's nout rows (WRAP: of all slabs; SEG: after the hbn halo rows) to
// the array.
template <class T, int U, int W, bool WRAP>
__device__ __forceinline__ void tile_store_w(T *base, const double *__restrict__ src, const TileArgs &a, int nout,
                                             int cbw, int hbn, int r0) {
    constexpr int UW = W == 1 ? U : U / 2;
    const int n1 = (int)a.p.n1, tid = (int)threadIdx.x, nthr = (int)blockDim.x, cb = a.cb;
    const unsigned cq = (unsigned)(cb / W), mq = W == 1 ? a.mcb : a.mcw;
    const i64 n2 = a.p.n2;
    const int total = nout * (int)cq;
#pragma unroll 1
    for (int q0 = tid; q0 < total; q0 += UW * nthr) {
#pragma unroll
        for (int i = 0; i < UW; ++i) {
            const unsigned q = (unsigned)(q0 + i * nthr);
            const unsigned row = cq == 1 ? q : __umulhi(q, mq);
            const unsigned col = (q - row * cq) * W;
            if ((int)row < nout && (int)col < cbw) {
                const double *w;
                T *dst;
                if constexpr (WRAP) {
                    const unsigned s = __umulhi(row, a.mn1);
                    w = src + (int)(s * (unsigned)cb + col) * a.pl + (int)(row - s * (unsigned)n1);
                    dst = base + (i64)row * n2;
                } else {
                    w = src + (int)col * a.pl + hbn + (int)row;
                    dst = base + (i64)(r0 + (int)row) * n2;
                }
                TilePack<T, W> st;
#pragma unroll
                for (int k = 0; k < W; ++k) st.v[k] = (T)w[k * a.pl];
                *reinterpret_cast<TilePack<T, W> *>(dst + col) = st;
            }
        }
    }
}

template <class T, int U, bool WRAP>
__device__ __forceinline__ void tile_stage(const T *base, const T *__restrict__ hsrc, double *__restrict__ lds,
                                           const TileArgs &a, int nrow, int cbw, int hbn, int r0, int nr) {
    if (a.wide) tile_stage_w<T, U, 16 / sizeof(T), WRAP>(base, hsrc, lds, a, nrow, cbw, hbn, r0, nr);
    else tile_stage_w<T, U, 1, WRAP>(base, hsrc, lds, a, nrow, cbw, hbn, r0, nr);
}
template <class T, int U, bool WRAP>
__device__ __forceinline__ void tile_store(T *base, const double *__restrict__ src, const TileArgs &a, int nout, int cbw,
                                           int hbn, int r0) {
    if (a.wide) tile_store_w<T, U, 16 / sizeof(T), WRAP>(base, src, a, nout, cbw, hbn, r0);
    else tile_store_w<T, U, 1, WRAP>(base, src, a, nout, cbw, hbn, r0);
}

// Six-tap sum over w[0..5], from 0. on as the reference's: 0. + -0. is 0., so
// the first product is fused with 0. (at no cost).
template <bool FUSED> __device__ __forceinline__ double tile_taps(const double (&c)[6], const double *w) {
    double acc = fma(c[0], w[0], 0.0);
#pragma unroll
    for (int k = 1; k < 6; ++k) {
        if constexpr (FUSED)
            acc = fma(c[k], w[k], acc);
        else
            acc = acc + c[k] * w[k];
    }
    return acc;
}

template <class T, bool FUSED, bool RND, int V, bool WRAP>
__device__ __forceinline__ void tile_unit(T *__restrict__ data, const T *__restrict__ halo, const TileArgs &a, i64 unit,
                                          double *__restrict__ lds) {
    constexpr int E = kTileRows;
    if constexpr (!WRAP) lds += kTileLow;
    const int n1 = (int)a.p.n1;
    const i64 n2 = a.p.n2;
    const int tid = (int)threadIdx.x;
    const int cb = a.cb, pl = a.pl, ns = a.ns;

    // ---- the tile ----
    const i64 grp = unit / a.nct;
    const i64 col0 = (unit - grp * a.nct) * cb;
    const int cbw = (int)min((i64)cb, n2 - col0);
    i64 i0b;       // first slab
    int nsl = 1;   // slabs
    int nrow;      // rows staged (all slabs)
    int hbn = 0, r0 = 0, nr = 0;
    const T *hsrc = nullptr;
    if constexpr (WRAP) {
        i0b = a.s0 + grp * a.sb;
        nsl = (int)min((i64)a.sb, a.s1 - i0b);
        nrow = nsl * n1;
    } else {
        i0b = a.s0 + grp / a.nseg;
        const TileSeg s = tile_segment(a, i0b, (int)(grp % a.nseg));
        if (s.nr <= 0) return;  // uniform over the work-group
        hbn = ns * s.hb;
        r0 = s.r0;
        nr = s.nr;
        nrow = hbn + nr + ns * s.ha;
        hsrc = halo + grp * a.hrows * n2 + col0;
    }
    T *base = data + i0b * n1 * n2 + col0;

    tile_stage<T, E, WRAP>(a.apart ? halo + i0b * n1 * n2 + col0 : base, hsrc, lds, a, nrow, cbw, hbn, r0, nr);
    __builtin_amdgcn_sched_barrier(0);

    // ---- this thread's rows: feet, coefficients, window position ----
    const int c = tid / a.rt, g = tid - c * a.rt;
    const int sl = c / a.ct, cc = c - sl * a.ct;
    const bool act = sl < nsl && cc < cbw;
    const int half = n1 / 2;
    double coef[E][6];
    int d0 = 0;
    int turn = 0;  // rows whose shift differs from the first row's: two bits per row, 1 + shift - d0 (0: the same)
#pragma unroll
    for (int j = 0; j < E; ++j) {
        int lr = g * E + j;
        bool in = act;
        if constexpr (WRAP) {
            in = act && lr < n1;
        } else {
            lr += r0 - hbn;
            if (lr < 0) lr += n1;
            if (lr >= n1) lr -= n1;
        }
        double d_prev1 = 2.0;
        int d = in ? lr - tile_foot(a.p, (int)(i0b + sl), lr, d_prev1) : d0;
        adv_lag_basis(d_prev1, coef[j]);
        if (in && d > half) d -= n1;
        if (in && d < -half) d += n1;
        if (j == 0) d0 = d;
        if (d != d0) turn |= (d > d0 ? 2 : 3) << (2 * j);  // two adjacent shifts at most
        __builtin_amdgcn_sched_barrier(0);  // one row's temporaries at a time
    }
    int rb = g * E - d0 - 2;
    if constexpr (WRAP) {
        if (rb < 0) rb += n1;
        if (rb >= n1) rb -= n1;
    } else {
        rb = min(max(rb, 1 - kTileLow), a.rows - 1);  // beyond: every row of the thread is discarded
    }
    __syncthreads();

    // ---- steps ----
    const int plane = (sl * cb + cc) * pl;
    const int vstep = a.ct * pl;
    const int nv = (cbw + a.ct - 1) / a.ct;  // columns per thread in this tile (uniform)
    double *src = lds;                       // V = 1: two buffers in turn, one barrier per step
    double *alt = lds + a.sb * cb * pl;
    // o = the step's results of this thread's rows of the column whose window
    // starts at w0 (row rb)
    auto column = [&](const double *w0, double (&o)[E]) __attribute__((always_inline)) {
        if (turn == 0) {
            double w[kTileWin];
#pragma unroll
            for (int t = 0; t < kTileWin; ++t) w[t] = w0[t];
#pragma unroll
            for (int j = 0; j < E; ++j) o[j] = tile_taps<FUSED>(coef[j], w + j);
        } else {
            int tb = turn, r = rb;
            asm volatile("" : "+v"(tb), "+v"(r));  // nothing of this rare form is kept across the steps
#pragma unroll
            for (int j = 0; j < E; ++j) {
                const int t = (tb >> (2 * j)) & 3;
                int b = j - (t == 2 ? 1 : t == 3 ? -1 : 0);
                if (WRAP && r + b < 0) b += n1;
                double w[6];
#pragma unroll
                for (int k = 0; k < 6; ++k) w[k] = w0[b + k];
                o[j] = tile_taps<FUSED>(coef[j], w);
            }
        }
        if constexpr (RND) {
#pragma unroll
            for (int j = 0; j < E; ++j) o[j] = (double)(float)o[j];
        }
    };
    // Results to the thread's rows at dst, the first rows also after the last.
    const int left = WRAP ? n1 - g * E : E;  // rows of the line from this thread's first on
    auto put = [&](double *dst, const double (&o)[E]) __attribute__((always_inline)) {
        if (left >= E) {
#pragma unroll
            for (int j = 0; j < E; ++j) dst[j] = o[j];
        } else {
#pragma unroll
            for (int j = 0; j < E - 1; ++j)
                if (j < left) dst[j] = o[j];
        }
        if constexpr (WRAP) {
            if (g * E < kTileGhost) {
#pragma unroll
                for (int j = 0; j < E; ++j) dst[n1 + j] = o[j];
            }
        }
    };
    for (int s = 0; s < ns; ++s) {
        double o[E];
        if constexpr (V == 1) {
            if (act) {
                column(src + plane + rb, o);
                put(alt + plane + g * E, o);
            }
            __syncthreads();
            double *t = src;
            src = alt;
            alt = t;
        } else {
            // a column is written while the next one is read: one barrier
            // per column separates its reads from its writes
            double *w = lds + plane + g * E;
            const int shift = rb - g * E;
            int col = act ? cc : cbw;
#pragma unroll 1
            for (int v = 0; v < nv; ++v) {
                const bool on = col < cbw;
                if (on) column(w + shift, o);
                __syncthreads();
                if (on) put(w, o);
                w += vstep;
                col += a.ct;
            }
            if (nv == 1) __syncthreads();
        }
    }
    if constexpr (V > 1) __syncthreads();

    tile_store<T, E, WRAP>(base, src, a, WRAP ? nrow : nr, cbw, hbn, r0);
}

// Launch shape of the slabs [a.s0, a.s1) of one problem (host side).
struct TileShape {
    TileArgs a{};
    int e = 0;  // 0: the LDS form (below: V columns per thread); else the strip form with e rows per lane
    int v = 1;
    bool wrap = true;
    int threads = 0;
    u64 lds_bytes = 0;
    u64 halo_bytes = 0;  // SEG: snapshot buffer
};

// The LDS tile of the slabs [s0, s1) of a problem for passes of at most ns
// steps (ns = 0: chosen here, and returned in a.ns).  False where it does not
// fit: lines shorter than 16 rows, or whose halos leave too few rows of a
// segment.  whole_only: whole lines only, which need no snapshot.
bool tile_shape(const bkma_adv_params &p, u64 s0, u64 s1, u64 elem_size, int ns, u64 lds_max, TileShape *out,
                bool whole_only = false);
// The strip tile (adv_strip.hpp) of slabs whose shifts it covers.
bool strip_shape(const bkma_adv_params &p, u64 s0, u64 s1, u64 elem_size, int ns, u64 lds_max, TileShape *out);
// A problem's tiles for passes of ns steps (0: chosen here; the same for all
// parts, in parts[0].a.ns): with `strips`, strips for the slabs whose shifts
// they cover (first in the list, if there are any) and LDS tiles for the
// others.  Empty where there are none (tile_covers among the reasons).
std::vector<TileShape> tile_parts(const bkma_adv_params &p, u64 elem_size, int ns, u64 lds_max, bool strips);

// Work-groups of `threads` threads that one launch may have (HIP counts threads
// in 32 bits; the snapshots' work-groups have up to 256).
inline i64 tile_launch_units(int threads) { return 0xffffffffLL / std::max(threads, 256); }
// Slabs of a shape, cut into nseg segments each, that one launch may cover.
inline i64 tile_slabs_per_launch(const TileShape &sh, int nseg) {
    const i64 units = tile_launch_units(sh.threads) / sh.a.nct;
    return std::max<i64>(1, sh.wrap ? units * sh.a.sb : units / nseg);
}

// One pass of ns steps (at most the shape's).  `fused`: fused sums (FP32
// storage), `rnd`: rounded to FP32 after every step.  `from`: the array to read
// (of the same extents; no snapshot), else `data` in place.
bkma_status launch_tile(const TileShape &sh, bkma_dtype dt, bool fused, bool rnd, void *data, void *halo, int ns,
                        hipStream_t s, void *from = nullptr);

// Several problems' parts in one launch (ragged batches): tiles of one kind.
struct TileProblem {
    TileArgs a;
    void *data;
    void *halo;
    i64 first;        // first work-group of the problem
    i64 first_halo;   // SEG: first work-group of its snapshot
};
struct TileGroup {
    int e = 0, v = 1;
    bool wrap = true;
    int threads = 0;
    u64 lds_bytes = 0;
    int ns = 1;                     // steps per pass
    int count = 0;                  // problems
    i64 units = 0, halo_units = 0;  // work-groups
    TileProblem *table = nullptr;   // device
};
// One pass of ns steps (at most the group's) of every problem of the group.
bkma_status launch_tile_group(const TileGroup &g, bkma_dtype dt, bool rnd, int ns, hipStream_t s);

// The strip kernels (strip_f64.hip, strip_f32.hip, strip_f32_round.hip).
bkma_status launch_strip_f64(const TileShape &sh, const TileArgs &a, void *data, void *halo, hipStream_t s);
bkma_status launch_strip_f32(const TileShape &sh, const TileArgs &a, void *data, void *halo, hipStream_t s);
bkma_status launch_strip_f32_round(const TileShape &sh, const TileArgs &a, void *data, void *halo, hipStream_t s);
bkma_status launch_strip_group_f64(const TileGroup &g, int ns, hipStream_t s);
bkma_status launch_strip_group_f32(const TileGroup &g, int ns, hipStream_t s);
bkma_status launch_strip_group_f32_round(const TileGroup &g, int ns, hipStream_t s);

// Consecutive tiles of one memory line (the column tiles of a slab) on one
// XCD: work-groups go to the 8 XCDs in turn.
__device__ __forceinline__ i64 tile_of_block(i64 b, i64 units, int nct) {
    const i64 per = units / 8;
    return nct > 1 && b < per * 8 ? (b % 8) * per + b / 8 : b;
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

// Allows the whole LDS to the kernel, once per device.
template <class K> bkma_status allow_lds(K kernel, std::atomic<unsigned> &done) {
    int dev = 0;
    BKMA_HIP_TRY(hipGetDevice(&dev));
    const unsigned bit = 1u << (dev & 31);
    if (done.load(std::memory_order_relaxed) & bit) return BKMA_OK;
    u64 lds_max = 0;
    BKMA_TRY(lds_limit_bytes(&lds_max));
    BKMA_HIP_TRY(hipFuncSetAttribute((const void *)kernel, hipFuncAttributeMaxDynamicSharedMemorySize, (int)lds_max));
    done.fetch_or(bit, std::memory_order_relaxed);
    return BKMA_OK;
}

}  // namespace bkma
