// FP64 and FP32 Conv1d, textbook semantics, in place (see bkma_conv.hip):
//   y[b][oc][j] = bias[oc] + sum_ic sum_k w[oc][ic][k] x[b][ic][j + k].
//
// A tile of TN columns of one batch element is staged in LDS with the K-1
// columns after it, then every output channel of it is computed and stored;
// an owner (a wavefront, two, or a work-group) takes a chunk of consecutive
// tiles in increasing order, so the columns after a tile are still unwritten
// as far as the chunk goes.  The K-1 columns after a chunk belong to another
// owner: they are copied first, and every tile that reaches past its chunk (with
// K-1 > TN not only the last) takes them from the copy.
//
// conv_valu_kernel (FP64; FP32 with few channels).  A lane holds JT columns
// and OCB output channels of its wave's channel group.  The weights of a tap
// are the same for the whole wave, so they are scalar loads and scalar
// operands; an LDS read of x feeds OCB channels.  FP64 keeps the oracle's
// order (bias, then ic, then k) and its separate multiply and add, so it is
// held at half the FP64 FMA rate; FP32 fuses them.
//   Before: weights from global memory per lane, 4 channels x 8 columns per
//   thread and 32 channel blocks per work-group whatever C: with C = 6 two
//   threads of 32 worked.  [16384][6][256], K = 5, FP64: 1734 -> 126 us.
//
// conv_lane64_kernel (FP64, C >= 17 and the common K).  A lane holds one
// channel and 16 columns, so a weight is a coalesced vector load and x an LDS
// broadcast; the wave-uniform weights of the form above come from L2 once they
// pass the 16 KB scalar cache, and a wait for LDS waits for them too
// ([256][128][4096], K = 5: 18.4 ms with it, 6.9 ms = 24.8 TFLOP/s here).
//
// conv_mfma32_kernel (FP32, 12 channels and more but for some that pad much).  v_mfma_f32_16x16x4_f32 keeps FP32
// products and sums (partial sums of 160 products are added up separately: the
// error against FP64 is half that of one long FP32 sum); its rate is twice that of the VALU without packed math.
// Waves split the output channels (blocks of 16) and, when there are few, the
// columns of a tile.  An operand is one VGPR per 32 cycles of matrix work, so
// weights stream from L2 and x is read from LDS one value per lane and MFMA;
// LDS rows start 16 banks apart, which spreads the four rows of an operand
// over all 64 banks.  [256][128][4096], K = 5: 14.0 -> 1.53 ms
//   (112 TFLOP/s, the matrix cores 65-75% busy: a tile is staged while only
//   the CU's other work-group computes).
#include <algorithm>
#include <new>
#include <utility>

#include "conv_direct.hpp"

namespace bkma {

constexpr int kMfmaBlock = 40;  // steps (160 products) to a partial sum
constexpr int kMfmaPad = 3;  // steps of the packed weights read ahead of the last

typedef float f32x4_t __attribute__((ext_vector_type(4)));

// Weights of the VALU form: [group][ic][k][OCB], zero past C.
template <class T>
__global__ void conv_pack_valu_kernel(const T *__restrict__ w, int C, int K, int ocb, i64 total, T *__restrict__ out) {
    for (i64 i = (i64)blockIdx.x * blockDim.x + threadIdx.x; i < total; i += (i64)gridDim.x * blockDim.x) {
        const int o = (int)(i % ocb);
        const i64 r = i / ocb;
        const int k = (int)(r % K);
        const int ic = (int)((r / K) % C);
        const int oc = (int)(r / ((i64)K * C)) * ocb + o;
        out[i] = oc < C ? w[((i64)oc * C + ic) * K + k] : (T)0;
    }
}

// Weights of the matrix form: [group][ic/4][k][MB][lane], lane l holding
// channel 16 (MB group + m) + l%16, input channel 4 i + l/16; zero past C.
__global__ void conv_pack_mfma32_kernel(const float *__restrict__ w, int C, int K, int mb, i64 total,
                                        float *__restrict__ out) {
    const int c4 = (C + 3) / 4;
    for (i64 i = (i64)blockIdx.x * blockDim.x + threadIdx.x; i < total; i += (i64)gridDim.x * blockDim.x) {
        const int l = (int)(i % 64);
        i64 r = i / 64;
        const int m = (int)(r % mb);
        r /= mb;
        const int k = (int)(r % K);
        r /= K;
        const int ic = 4 * (int)(r % c4) + l / 16;
        const int oc = 16 * ((int)(r / c4) * mb + m) + l % 16;
        out[i] = oc < C && ic < C ? w[((i64)oc * C + ic) * K + k] : 0.0f;
    }
}

// The K-1 columns after every chunk (none where it ends with a row).
template <class T>
__global__ void conv_owner_halo_kernel(const T *__restrict__ x, T *__restrict__ halo, int C, int L, int K, int TN,
                                       int tiles, int total, int chunk) {
    const int c = blockIdx.x;
    const ConvChunk ck = conv_chunk(c, chunk, total);
    if (ck.end <= ck.first) return;
    const int b = (ck.end - 1) / tiles, j0 = ck.column_after(b, tiles, TN);
    if (j0 == 0x7fffffff) return;
    const int H = K - 1;
    for (int e = threadIdx.x; e < C * H; e += blockDim.x) {
        const int ic = e / H, kk = e - ic * H;
        const int j = j0 + kk;
        halo[(i64)c * C * H + e] = j < L ? x[((i64)b * C + ic) * L + j] : (T)0;
    }
}

// Stages one tile: rows [0, rows), columns [0, TN + H), zero past the row end
// and for rows past C.  `t` of `nt` threads; TN is a power of two (1 << tsh);
// vec: 16-byte loads (rows and the array on 16-byte boundaries).
template <class T, bool VEC>
__device__ __forceinline__ void stage_columns(const T *__restrict__ xb, T *__restrict__ xs, int C, int rows, int L,
                                              int j0, int tsh, int pitch, int t, int nt) {
    constexpr int N = VEC ? 16 / (int)sizeof(T) : 1, U = VEC ? 8 : 16;  // elements per load, loads in flight
    constexpr int SH = N == 4 ? 2 : N == 2 ? 1 : 0;
    using VT = T __attribute__((ext_vector_type(N)));
    const int per = tsh - SH, items = rows << per, mask = (1 << per) - 1;
    for (int i0 = t; i0 < items; i0 += U * nt) {
        VT v[U];
#pragma unroll
        for (int u = 0; u < U; ++u) {
            const int i = i0 + u * nt, row = i >> per, col = (i & mask) << SH;
            v[u] = (VT)(T)0;
            // L is a multiple of N: a piece lies inside the row or past it
            if (i < items && row < C && j0 + col < L) v[u] = *reinterpret_cast<const VT *>(xb + (i64)row * L + j0 + col);
        }
#pragma unroll
        for (int u = 0; u < U; ++u) {
            const int i = i0 + u * nt, row = i >> per, col = (i & mask) << SH;
            if (i < items) {
#pragma unroll
                for (int c = 0; c < N; ++c) xs[row * pitch + col + c] = v[u][c];
            }
        }
    }
}

// hsnap: the owner's copy of the row's columns from jend on, which come after its chunk.
template <class T>
__device__ __forceinline__ void stage_tile(const T *__restrict__ xb, const T *__restrict__ hsnap, int jend,
                                           T *__restrict__ xs, int C, int rows, int L, int j0, int tsh, int H,
                                           int pitch, bool vec, int t, int nt) {
    const int TN = 1 << tsh;
    // the H columns after the tile, from the snapshot or the row
    for (int e = t; e < rows * H; e += nt) {
        const int row = e / H, col = e - row * H, j = j0 + TN + col;
        T v = (T)0;
        if (row < C) {
            if (j >= jend) v = hsnap[row * H + (j - jend)];
            else if (j < L) v = xb[(i64)row * L + j];
        }
        xs[row * pitch + TN + col] = v;
    }
    if (vec) stage_columns<T, true>(xb, xs, C, rows, L, j0, tsh, pitch, t, nt);
    else stage_columns<T, false>(xb, xs, C, rows, L, j0, tsh, pitch, t, nt);
}

template <class T, int OCB, int JT>
__global__ __launch_bounds__(256) void conv_valu_kernel(T *__restrict__ x, const T *__restrict__ halo,
                                                        const T *__restrict__ wpk, const T *__restrict__ bias, int C,
                                                        int L, int K, int tiles, int total, int chunk, int wpt,
                                                        int groups, int pitch, bool vec) {
    extern __shared__ __align__(16) unsigned char conv_lds[];
    constexpr int TN = 64 * JT;
    const int lane = threadIdx.x & 63;
    const int wave = __builtin_amdgcn_readfirstlane((int)(threadIdx.x >> 6));
    const int slot = wave / wpt, ws = wave - slot * wpt;
    const int owner = (int)blockIdx.x * (4 / wpt) + slot;
    T *xs = reinterpret_cast<T *>(conv_lds) + (i64)slot * C * pitch;
    const int Lout = L - K + 1;
    const ConvChunk ck = conv_chunk(owner, chunk, total);
    for (int it = 0; it < chunk; ++it) {  // the same count for all waves: the barriers are uniform
        const bool on = it < ck.end - ck.first;
        const int tile = on ? ck.first + it : 0;
        const int b = tile / tiles, t = tile - b * tiles;
        const int j0 = t * TN;
        T *xb = x + (i64)b * C * L;
        if (on) {
            stage_tile(xb, halo + (i64)owner * C * (K - 1), ck.column_after(b, tiles, TN), xs, C, C, L, j0,
                       JT == 4 ? 8 : JT == 2 ? 7 : 6, K - 1, pitch, vec, ws * 64 + lane, wpt * 64);
        }
        __syncthreads();
        if (on) {
            for (int g = ws; g < groups; g += wpt) {
                T acc[OCB][JT];
                const T *wp = wpk + (i64)g * C * K * OCB;
#pragma unroll
                for (int o = 0; o < OCB; ++o) {
                    const int oc = g * OCB + o;
                    const T bv = bias[oc < C ? oc : C - 1];
#pragma unroll
                    for (int c = 0; c < JT; ++c) acc[o][c] = bv;
                }
                for (int ic = 0; ic < C; ++ic) {
                    const T *xr = xs + ic * pitch + lane;
#pragma unroll 2
                    for (int k = 0; k < K; ++k) {
                        T wv[OCB];
#pragma unroll
                        for (int o = 0; o < OCB; ++o) wv[o] = wp[o];
                        wp += OCB;
                        T xv[JT];
#pragma unroll
                        for (int c = 0; c < JT; ++c) xv[c] = xr[64 * c + k];
#pragma unroll
                        for (int o = 0; o < OCB; ++o)
#pragma unroll
                            for (int c = 0; c < JT; ++c) {
                                if constexpr (sizeof(T) == 8) acc[o][c] = acc[o][c] + wv[o] * xv[c];
                                else acc[o][c] = __builtin_fmaf(wv[o], xv[c], acc[o][c]);
                            }
                    }
                }
#pragma unroll
                for (int o = 0; o < OCB; ++o) {
                    const int oc = g * OCB + o;
                    if (oc < C) {
#pragma unroll
                        for (int c = 0; c < JT; ++c) {
                            const int j = j0 + lane + 64 * c;
                            if (j < Lout) xb[(i64)oc * L + j] = acc[o][c];
                        }
                    }
                }
            }
        }
        __syncthreads();
    }
}

// FP64 with many channels: a lane holds one output channel and kLaneCols
// columns; CW lanes span the channels of a group, the 64 / CW parts of a
// wavefront take neighbouring columns.  x is the same for the lanes of a part
// (one LDS read of two columns feeds all taps through a register window),
// the weights are a coalesced vector load per tap, one input channel ahead.
constexpr int kLaneCols = 16;

// Weights of the lane form: [group][ic][k][CW], zero past C.
template <int KT>
__global__ __launch_bounds__(256) void conv_lane64_kernel(double *__restrict__ x, const double *__restrict__ halo,
                                                          const double *__restrict__ wpk,
                                                          const double *__restrict__ bias, int C, int L, int tiles,
                                                          int total, int chunk, int groups, int cw, int tsh, int pitch,
                                                          bool vec) {
    extern __shared__ __align__(16) unsigned char conv_lds[];
    double *xs = reinterpret_cast<double *>(conv_lds);
    constexpr int JT = kLaneCols, W = (JT + KT - 1 + 1) & ~1;  // window, whole pairs
    const int lane = threadIdx.x & 63;
    const int wave = __builtin_amdgcn_readfirstlane((int)(threadIdx.x >> 6));
    const int TN = 1 << tsh, Lout = L - KT + 1;
    const int ol = lane & (cw - 1), part = lane / cw;
    const int span = JT * (64 / cw);  // columns of a wavefront
    const int blocks = TN / span;
    const ConvChunk ck = conv_chunk((int)blockIdx.x, chunk, total);
    for (int tile = ck.first; tile < ck.end; ++tile) {
        const int b = tile / tiles, t = tile - b * tiles;
        const int j0 = t * TN;
        double *xb = x + (i64)b * C * L;
        stage_tile(xb, halo + (i64)blockIdx.x * C * (KT - 1), ck.column_after(b, tiles, TN), xs, C, C, L, j0, tsh,
                   KT - 1, pitch, vec, (int)threadIdx.x, 256);
        __syncthreads();
        for (int item = wave; item < groups * blocks; item += 4) {
            const int g = item / blocks, blk = item - g * blocks;
            const int oc = g * cw + ol;
            const int jl = blk * span + part * JT;
            const double bv = bias[oc < C ? oc : C - 1];
            double acc[JT];
#pragma unroll
            for (int c = 0; c < JT; ++c) acc[c] = bv;
            const double *wp = wpk + (i64)g * C * KT * cw + ol;
            double wn[KT];
#pragma unroll
            for (int k = 0; k < KT; ++k) wn[k] = wp[k * cw];
            const double *xr = xs + jl;
            for (int ic = 0; ic < C; ++ic) {
                double wv[KT], xw[W];
#pragma unroll
                for (int k = 0; k < KT; ++k) wv[k] = wn[k];
                if (ic + 1 < C) wp += KT * cw;
#pragma unroll
                for (int k = 0; k < KT; ++k) wn[k] = wp[k * cw];
#pragma unroll
                for (int i = 0; i < W; i += 2) {
                    const double2 v = *reinterpret_cast<const double2 *>(xr + i);
                    xw[i] = v.x;
                    xw[i + 1] = v.y;
                }
                xr += pitch;
#pragma unroll
                for (int k = 0; k < KT; ++k)
#pragma unroll
                    for (int c = 0; c < JT; ++c) acc[c] = acc[c] + wv[k] * xw[c + k];
            }
            if (oc < C) {
                double *dst = xb + (i64)oc * L + j0 + jl;
#pragma unroll
                for (int c = 0; c < JT; ++c)
                    if (j0 + jl + c < Lout) dst[c] = acc[c];
            }
        }
        __syncthreads();
    }
}

// MB blocks of 16 channels, NB blocks of 16 columns per wave.
template <int MB, int NB>
__global__ __launch_bounds__(256) void conv_mfma32_kernel(float *__restrict__ x, const float *__restrict__ halo,
                                                          const float *__restrict__ wpk,
                                                          const float *__restrict__ bias, int C, int L, int K,
                                                          int tiles, int total, int chunk, int groups, int parts,
                                                          int tsh, int pitch, bool vec) {
    extern __shared__ __align__(16) unsigned char conv_lds[];
    float *xs = reinterpret_cast<float *>(conv_lds);
    const int lane = threadIdx.x & 63;
    const int wave = __builtin_amdgcn_readfirstlane((int)(threadIdx.x >> 6));
    const int TN = 1 << tsh, Lout = L - K + 1;
    const int c4 = (C + 3) / 4, steps = c4 * K;
    const int lc = lane & 15, lr = lane >> 4;
    const ConvChunk ck = conv_chunk((int)blockIdx.x, chunk, total);
    for (int tile = ck.first; tile < ck.end; ++tile) {
        const int b = tile / tiles, t = tile - b * tiles;
        const int j0 = t * TN;
        float *xb = x + (i64)b * C * L;
        stage_tile(xb, halo + (i64)blockIdx.x * C * (K - 1), ck.column_after(b, tiles, TN), xs, C, 4 * c4, L, j0, tsh,
                   K - 1, pitch, vec, (int)threadIdx.x, 256);
        __syncthreads();
        for (int item = wave; item < groups * parts; item += 4) {
            const int g = item / parts, part = item - g * parts;
            const float *wp = wpk + (i64)g * steps * MB * 64 + lane;
            const float *xr = xs + lr * pitch + part * 16 * NB + lc;
            f32x4_t acc[MB][NB], sum[MB][NB];
#pragma unroll
            for (int m = 0; m < MB; ++m)
#pragma unroll
                for (int r = 0; r < 4; ++r) {
                    const int oc = 16 * (g * MB + m) + 4 * lr + r;
                    const float bv = bias[oc < C ? oc : C - 1];
#pragma unroll
                    for (int n = 0; n < NB; ++n) {
                        sum[m][n][r] = bv;
                        acc[m][n][r] = 0.0f;
                    }
                }
            // Weights three steps and x one step ahead, in registers that
            // rotate by unrolling (a move out of a load's destination would
            // wait for it); the packed array ends in kAhead steps of padding.
            constexpr int kAhead = kMfmaPad;
            float aw[kAhead + 1][MB], bx[2][NB];
#pragma unroll
            for (int u = 0; u < kAhead; ++u)
#pragma unroll
                for (int m = 0; m < MB; ++m) aw[u][m] = wp[(u * MB + m) * 64];
            wp += kAhead * MB * 64;
            int k = 0;
#pragma unroll
            for (int n = 0; n < NB; ++n) bx[0][n] = xr[16 * n];
            for (int s0 = 0; s0 < steps; s0 += kAhead + 1) {
                static_for<0, kAhead + 1>([&](auto u_) __attribute__((always_inline)) {
                    constexpr int u = decltype(u_)::value;
                    const int s = s0 + u;
                    if (s >= steps) return;
#pragma unroll
                    for (int m = 0; m < MB; ++m) aw[(u + kAhead) % (kAhead + 1)][m] = wp[m * 64];
                    wp += MB * 64;
                    // next tap, or the first tap of the next four input
                    // channels (after the last step: the same place again)
                    if (++k == K) {
                        k = 0;
                        xr += s + 1 < steps ? 4 * pitch - (K - 1) : 0;
                    } else {
                        xr += 1;
                    }
#pragma unroll
                    for (int n = 0; n < NB; ++n) bx[(u + 1) % 2][n] = xr[16 * n];
                    __builtin_amdgcn_sched_barrier(0);
#pragma unroll
                    for (int n = 0; n < NB; ++n)
#pragma unroll
                        for (int m = 0; m < MB; ++m)
                            acc[m][n] = __builtin_amdgcn_mfma_f32_16x16x4f32(aw[u][m], bx[u % 2][n], acc[m][n], 0, 0, 0);
                    __builtin_amdgcn_sched_barrier(0);
                });
                // sums of kMfmaBlock steps are added up separately: the
                // roundings of one long sum would be twice as large
                if ((s0 + kAhead + 1) % kMfmaBlock == 0 || s0 + kAhead + 1 >= steps) {
#pragma unroll
                    for (int m = 0; m < MB; ++m)
#pragma unroll
                        for (int n = 0; n < NB; ++n) {
                            sum[m][n] += acc[m][n];
                            acc[m][n] = (f32x4_t)0.0f;
                        }
                }
            }
            // D[row][col]: lane l, register r holds row 4 (l/16) + r, column l%16
#pragma unroll
            for (int m = 0; m < MB; ++m)
#pragma unroll
                for (int r = 0; r < 4; ++r) {
                    const int oc = 16 * (g * MB + m) + 4 * lr + r;
                    if (oc < C) {
#pragma unroll
                        for (int n = 0; n < NB; ++n) {
                            const int j = j0 + part * 16 * NB + 16 * n + lc;
                            if (j < Lout) xb[(i64)oc * L + j] = sum[m][n][r];
                        }
                    }
                }
        }
        __syncthreads();
    }
}

// ---------------------------------------------------------------------------
// Host side
// ---------------------------------------------------------------------------
namespace {

template <class T, int OCB, int JT> const void *valu_kernel() { return (const void *)conv_valu_kernel<T, OCB, JT>; }

template <class T, int OCB> const void *valu_kernel_jt(int jt) {
    return jt == 4 ? valu_kernel<T, OCB, 4>() : jt == 2 ? valu_kernel<T, OCB, 2>() : valu_kernel<T, OCB, 1>();
}

template <class T> const void *valu_kernel_of(int ocb, int jt) {
    switch (ocb) {
        case 8: return valu_kernel_jt<T, 8>(jt);
        case 6: return valu_kernel_jt<T, 6>(jt);
        case 5: return valu_kernel_jt<T, 5>(jt);
        case 4: return valu_kernel_jt<T, 4>(jt);
        case 3: return valu_kernel_jt<T, 3>(jt);
        case 2: return valu_kernel_jt<T, 2>(jt);
        default: return valu_kernel_jt<T, 1>(jt);
    }
}

const void *mfma_kernel_of(int mb, int nb) {
    if (mb == 2)
        return nb == 8 ? (const void *)conv_mfma32_kernel<2, 8>
                       : nb == 4 ? (const void *)conv_mfma32_kernel<2, 4> : (const void *)conv_mfma32_kernel<2, 2>;
    if (mb == 3) return (const void *)conv_mfma32_kernel<3, 2>;  // one group: the waves split 128 columns
    return nb == 8 ? (const void *)conv_mfma32_kernel<1, 8>
                   : nb == 4 ? (const void *)conv_mfma32_kernel<1, 4> : (const void *)conv_mfma32_kernel<1, 2>;
}

const void *lane_kernel_of(int K) {
    switch (K) {
        case 1: return (const void *)conv_lane64_kernel<1>;
        case 2: return (const void *)conv_lane64_kernel<2>;
        case 3: return (const void *)conv_lane64_kernel<3>;
        case 4: return (const void *)conv_lane64_kernel<4>;
        case 5: return (const void *)conv_lane64_kernel<5>;
        case 7: return (const void *)conv_lane64_kernel<7>;
        case 9: return (const void *)conv_lane64_kernel<9>;
        case 11: return (const void *)conv_lane64_kernel<11>;
        default: return nullptr;
    }
}

const void *kernel_of(const DirectConv &d) {
    if (d.lane) return lane_kernel_of(d.K);
    if (d.mfma) return mfma_kernel_of(d.ocb, d.jt);
    return d.dt == BKMA_F64 ? valu_kernel_of<double>(d.ocb, d.jt) : valu_kernel_of<float>(d.ocb, d.jt);
}

}  // namespace

void direct_conv_free(DirectConv &d) {
    if (d.w) (void)hipFree(d.w);
    d.w = nullptr;
    d.halo.reset();
}

bkma_status direct_conv_create(bkma_dtype dt, int B, int C, int L, int K, const void *weight, hipStream_t s,
                               DirectConv *out) {
    DirectConv d;
    d.dt = dt;
    d.B = B;
    d.C = C;
    d.L = L;
    d.K = K;
    const u64 esz = dt == BKMA_F64 ? 8 : 4;
    const int Lout = L - K + 1;
    u64 lds_max = 0;
    BKMA_TRY(lds_limit_bytes(&lds_max));
    // FP32: the matrix cores where 16 channels, or 32, do not pad too much
    // ([B][C][1000], K = 5, matrix cores / VALU, us: C = 12 39 / 33, 16 33 / 42,
    // 17 55 / 40, 20 53 / 50, 24 51 / 55, 32 53 / 72)
    // (kernels so long that only the narrowest tile fits stay with it, and so do
    // few columns, [81][18][1152], K = 1: 7.3 / 11.9, and K = 3, 57 / 52 to 60 / 64)
    const bool pads = (C == 12 || (C >= 17 && C <= 20 && K >= 5)) && (u64)B * (u64)Lout >= (1u << 18);
    d.mfma = dt == BKMA_F32 && C >= 12 && (!pads || K > 1024);
    u64 wcount = 0;
    if (d.mfma) {
        d.ocb = C <= 16 ? 1 : C > 32 && C <= 48 && K <= 64 ? 3 : 2;  // three blocks of 16 channels instead of two times two
        d.groups = (int)ceil_div((u64)C, (u64)(16 * d.ocb));
        d.parts = d.groups >= 4 ? 1 : d.groups >= 2 ? 2 : 4;
        const u64 rows = ceil_div((u64)C, 4) * 4;
        // Tiles of 128, 64 or 32 columns (at most 8 blocks a wave): the rounds
        // of the resident work-groups, their share of a CU, the tile's columns
        // and what narrower tiles lose (weights are read once per tile).  FP32,
        // 128 -> 64 columns, us: [256][128][4096], K = 5: 1546 -> 1773;
        // [65][128][1000], 520 tiles of 128 on 512 work-groups: 208 -> 181;
        // [344][128][190], K = 1: 71 -> 55.
        int cus = 0, dev = 0;
        if (hipGetDevice(&dev) != hipSuccess ||
            hipDeviceGetAttribute(&cus, hipDeviceAttributeMultiprocessorCount, dev) != hipSuccess)
            return fail(BKMA_ERR_DEVICE, "conv1d plan: device query");
        double least = 0;
        // rows 16 banks apart modulo 64; where no tile fits so but the VALU form's
        // would, 48 apart, which also spreads an operand's four rows (32 columns
        // and K - 1 of 600 channels: 80 or 48 a row)
        for (const auto &[apart, tn] : {std::pair{16, 128}, {16, 64}, {16, 32}, {48, 32}}) {
            const int nb = tn / 16 / d.parts;
            if (nb > 8 || nb < 2) continue;
            if (tn > 32 && tn / 2 >= Lout && nb > 2) continue;  // half of the tile would stay empty
            if (apart == 48 && (d.TN || (u64)C * (u64)(64 + K - 1) * esz > lds_max)) continue;
            const int pitch = tn + K - 1 + ((apart - (tn + K - 1)) % 64 + 64) % 64;
            const u64 b = rows * (u64)pitch * esz;
            if (b > lds_max) continue;
            const void *kern = mfma_kernel_of(d.ocb, nb);
            int blocks = 0;
            if (hipFuncSetAttribute(kern, hipFuncAttributeMaxDynamicSharedMemorySize, (int)lds_max) != hipSuccess ||
                hipOccupancyMaxActiveBlocksPerMultiprocessor(&blocks, kern, 256, (size_t)b) != hipSuccess)
                return fail(BKMA_ERR_DEVICE, "conv1d plan: occupancy query");
            blocks = std::max(blocks, 1);
            const u64 all = ceil_div((u64)Lout, (u64)tn) * (u64)B;
            const double cost = (double)ceil_div(all, (u64)blocks * (u64)cus) * blocks * tn *
                                (tn == 128 ? 1.0 : tn == 64 ? 1.1 : 1.6) * (blocks == 1 ? 1.3 : 1.0);
            if (d.TN && cost >= least) continue;
            least = cost;
            d.TN = tn;
            d.jt = nb;
            d.pitch = pitch;
            d.lds_bytes = b;
        }
        if (!d.TN) d.mfma = false;  // too many channels for the padded tile
        wcount = ((u64)d.groups * (rows / 4) * K + kMfmaPad) * d.ocb * 64;
    }
    if (dt == BKMA_F64 && C >= 17 && lane_kernel_of(K)) {
        int cw = 64;
        while (cw > 16 && cw / 2 >= C) cw /= 2;
        const int span = kLaneCols * (64 / cw);
        const int groups = (int)ceil_div((u64)C, (u64)cw);
        for (int blocks = groups >= 4 ? 1 : groups >= 2 ? 2 : 4; blocks >= 1 && !d.lane; blocks /= 2) {
            const int tn = span * blocks, pitch = (tn + K - 1 + 2) & ~1;
            const u64 b = (u64)C * pitch * esz;
            if ((blocks > 1 && tn / 2 >= Lout) || b > lds_max) continue;
            d.lane = true;
            d.ocb = cw;
            d.groups = groups;
            d.TN = tn;
            d.pitch = pitch;
            d.lds_bytes = b;
        }
        wcount = (u64)d.groups * C * K * d.ocb;
    }
    if (!d.mfma && !d.lane) {
        // channels per thread: padded channels times what one of them costs, an
        // LDS read shared by o of them included (FP64 [2659][11][771], K = 5:
        // 239 us with one channel, 177 with six of twelve)
        int best = 0;
        double least = 0;
        for (int o : {8, 6, 5, 4, 3, 2, 1}) {
            const double cost = (double)((C + o - 1) / o * o) * (2.0 + 1.5 / o);
            if (best && cost >= least) continue;
            best = o;
            least = cost;
        }
        d.ocb = best;
        d.groups = (C + best - 1) / best;
        d.wpt = d.groups >= 4 ? 4 : d.groups >= 2 ? 2 : 1;
        d.TN = 0;
        for (u64 room : {lds_max / 3, lds_max / 2, lds_max}) {
            for (int jt : {4, 2, 1}) {
                if (d.TN || (jt > 1 && 32 * jt >= Lout)) continue;
                const int pitch = 64 * jt + K - 1;
                for (int wpt = d.wpt; wpt <= 4; wpt *= 2) {
                    const u64 b = (u64)(4 / wpt) * C * pitch * esz;
                    if (d.TN || b > room) continue;
                    d.TN = 64 * jt;
                    d.jt = jt;
                    d.wpt = wpt;
                    d.pitch = pitch;
                    d.lds_bytes = b;
                }
            }
        }
        if (!d.TN) return fail(BKMA_ERR_UNSUPPORTED, "conv1d plan: C too large for the LDS tile");
        wcount = (u64)d.groups * C * K * d.ocb;
    }
    const u64 tiles = ceil_div((u64)Lout, (u64)d.TN);
    if (tiles * (u64)B > 0x7fffffffULL) return fail(BKMA_ERR_UNSUPPORTED, "conv1d plan: sizes beyond 32-bit indexing");
    d.tiles = (int)tiles;
    d.total = (int)(tiles * B);
    d.slots = d.mfma || d.lane ? 1 : 4 / d.wpt;
    int dev = 0, cus = 0, blocks = 0;
    if (hipGetDevice(&dev) != hipSuccess ||
        hipDeviceGetAttribute(&cus, hipDeviceAttributeMultiprocessorCount, dev) != hipSuccess)
        return fail(BKMA_ERR_DEVICE, "conv1d plan: device query");
    const void *k = kernel_of(d);
    if (hipFuncSetAttribute(k, hipFuncAttributeMaxDynamicSharedMemorySize, (int)lds_max) != hipSuccess ||
        hipOccupancyMaxActiveBlocksPerMultiprocessor(&blocks, k, 256, (size_t)d.lds_bytes) != hipSuccess)
        return fail(BKMA_ERR_DEVICE, "conv1d plan: occupancy query");
    const u64 resident = (u64)std::max(1, blocks) * (u64)cus * (u64)d.slots;
    d.chunk = (int)ceil_div((u64)d.total, std::min<u64>((u64)d.total, resident));
    d.owners = (int)ceil_div((u64)d.total, (u64)d.chunk);
    d.grid = (unsigned)ceil_div((u64)d.owners, (u64)d.slots);
    bool room = hipMalloc(&d.w, wcount * esz) == hipSuccess;
    if (room && d.tiles > 1 && K > 1) {
        // for up to four streams and captures, within a quarter of x
        const u64 bytes = (u64)d.owners * C * (K - 1) * esz, quarter = (u64)B * C * L * esz / 4;
        d.halo.reset(new (std::nothrow) StreamScratch());
        room = d.halo && d.halo->create(bytes, bytes, (int)std::min<u64>(3, quarter / bytes));
    }
    if (!room) {
        direct_conv_free(d);
        return fail(BKMA_ERR_OUT_OF_MEMORY, "conv1d plan: weight copy");
    }
    if (d.mfma) {
        const u64 body = wcount - (u64)kMfmaPad * d.ocb * 64;
        hipLaunchKernelGGL(conv_pack_mfma32_kernel, dim3(256), dim3(256), 0, s, (const float *)weight, C, K, d.ocb,
                           (i64)body, (float *)d.w);
    } else if (dt == BKMA_F64) {
        hipLaunchKernelGGL(conv_pack_valu_kernel<double>, dim3(256), dim3(256), 0, s, (const double *)weight, C, K, d.ocb,
                           (i64)wcount, (double *)d.w);
    } else {
        hipLaunchKernelGGL(conv_pack_valu_kernel<float>, dim3(256), dim3(256), 0, s, (const float *)weight, C, K, d.ocb,
                           (i64)wcount, (float *)d.w);
    }
    if (hipGetLastError() != hipSuccess) {
        direct_conv_free(d);
        return fail(BKMA_ERR_DEVICE, "conv1d plan: weight packing");
    }
    *out = std::move(d);
    return BKMA_OK;
}

namespace {

int log2_of(int v) {
    int r = 0;
    while ((1 << r) < v) ++r;
    return r;
}

// Rows and array on 16-byte boundaries.
bool row_vec(const DirectConv &d, const void *x) {
    return reinterpret_cast<uintptr_t>(x) % 16 == 0 && ((u64)d.L * (d.dt == BKMA_F64 ? 8 : 4)) % 16 == 0;
}

// One run's share of the tiles.
struct ConvRun {
    int chunk = 0;
    unsigned grid = 0;
    void *halo = nullptr;
};

template <class T, int OCB, int JT>
void launch_valu(const DirectConv &d, const ConvRun &r, T *x, const T *bias, hipStream_t s) {
    hipLaunchKernelGGL((conv_valu_kernel<T, OCB, JT>), dim3(r.grid), dim3(256), (size_t)d.lds_bytes, s, x,
                       (const T *)r.halo, (const T *)d.w, bias, d.C, d.L, d.K, d.tiles, d.total, r.chunk, d.wpt,
                       d.groups, d.pitch, row_vec(d, x));
}

template <class T, int OCB>
void launch_valu_jt(const DirectConv &d, const ConvRun &r, T *x, const T *bias, hipStream_t s) {
    if (d.jt == 4) launch_valu<T, OCB, 4>(d, r, x, bias, s);
    else if (d.jt == 2) launch_valu<T, OCB, 2>(d, r, x, bias, s);
    else launch_valu<T, OCB, 1>(d, r, x, bias, s);
}

template <class T>
void launch_valu_of(const DirectConv &d, const ConvRun &r, T *x, const T *bias, hipStream_t s) {
    switch (d.ocb) {
        case 8: launch_valu_jt<T, 8>(d, r, x, bias, s); break;
        case 6: launch_valu_jt<T, 6>(d, r, x, bias, s); break;
        case 5: launch_valu_jt<T, 5>(d, r, x, bias, s); break;
        case 4: launch_valu_jt<T, 4>(d, r, x, bias, s); break;
        case 3: launch_valu_jt<T, 3>(d, r, x, bias, s); break;
        case 2: launch_valu_jt<T, 2>(d, r, x, bias, s); break;
        default: launch_valu_jt<T, 1>(d, r, x, bias, s); break;
    }
}

template <int MB, int NB>
void launch_mfma(const DirectConv &d, const ConvRun &r, float *x, const float *bias, hipStream_t s) {
    hipLaunchKernelGGL((conv_mfma32_kernel<MB, NB>), dim3(r.grid), dim3(256), (size_t)d.lds_bytes, s, x,
                       (const float *)r.halo, (const float *)d.w, bias, d.C, d.L, d.K, d.tiles, d.total, r.chunk,
                       d.groups, d.parts, log2_of(d.TN), d.pitch, row_vec(d, x));
}

template <int MB>
void launch_mfma_nb(const DirectConv &d, const ConvRun &r, float *x, const float *bias, hipStream_t s) {
    if (d.jt == 8) launch_mfma<MB, 8>(d, r, x, bias, s);
    else if (d.jt == 4) launch_mfma<MB, 4>(d, r, x, bias, s);
    else launch_mfma<MB, 2>(d, r, x, bias, s);
}

template <int KT>
void launch_lane_k(const DirectConv &d, const ConvRun &r, double *x, const double *bias, hipStream_t s) {
    hipLaunchKernelGGL(conv_lane64_kernel<KT>, dim3(r.grid), dim3(256), (size_t)d.lds_bytes, s, x,
                       (const double *)r.halo, (const double *)d.w, bias, d.C, d.L, d.tiles, d.total, r.chunk,
                       d.groups, d.ocb, log2_of(d.TN), d.pitch, row_vec(d, x));
}

bkma_status launch_lane(const DirectConv &d, const ConvRun &r, double *x, const double *bias, hipStream_t s) {
    switch (d.K) {
        case 1: launch_lane_k<1>(d, r, x, bias, s); break;
        case 2: launch_lane_k<2>(d, r, x, bias, s); break;
        case 3: launch_lane_k<3>(d, r, x, bias, s); break;
        case 4: launch_lane_k<4>(d, r, x, bias, s); break;
        case 5: launch_lane_k<5>(d, r, x, bias, s); break;
        case 7: launch_lane_k<7>(d, r, x, bias, s); break;
        case 9: launch_lane_k<9>(d, r, x, bias, s); break;
        case 11: launch_lane_k<11>(d, r, x, bias, s); break;
        default: return fail(BKMA_ERR_RUNTIME, "conv1d run: no lane kernel for this K");
    }
    return check_launch("conv_lane64_kernel");
}

template <class T> bkma_status run_direct(const DirectConv &d, T *x, const T *bias, hipStream_t s) {
    ConvRun r{d.chunk, d.grid, nullptr};
    std::unique_lock<std::mutex> held;
    if (d.halo) {
        held = d.halo->lock();
        r.halo = d.halo->get(s, false);
        if (r.halo) {
            hipLaunchKernelGGL(conv_owner_halo_kernel<T>, dim3((unsigned)d.owners), dim3(256), 0, s, (const T *)x,
                               (T *)r.halo, d.C, d.L, d.K, d.TN, d.tiles, d.total, d.chunk);
            BKMA_TRY(check_launch("conv_owner_halo_kernel"));
        } else {
            // no copy for this stream: chunks of whole rows, which need none
            r.chunk = (int)std::min<u64>((u64)d.total, ceil_div((u64)d.chunk, (u64)d.tiles) * (u64)d.tiles);
            r.grid = (unsigned)ceil_div(ceil_div((u64)d.total, (u64)r.chunk), (u64)d.slots);
        }
    }
    if constexpr (sizeof(T) == 4) {
        if (d.mfma) {
            if (d.ocb == 3) launch_mfma<3, 2>(d, r, x, bias, s);
            else if (d.ocb == 2) launch_mfma_nb<2>(d, r, x, bias, s);
            else launch_mfma_nb<1>(d, r, x, bias, s);
            return check_launch("conv_mfma32_kernel");
        }
    }
    if constexpr (sizeof(T) == 8) {
        if (d.lane) return launch_lane(d, r, x, bias, s);
    }
    launch_valu_of<T>(d, r, x, bias, s);
    return check_launch("conv_valu_kernel");
}

}  // namespace

bkma_status direct_conv_run(const DirectConv &d, void *x, const void *bias, hipStream_t s) {
    return d.dt == BKMA_F64 ? run_direct<double>(d, (double *)x, (const double *)bias, s)
                            : run_direct<float>(d, (float *)x, (const float *)bias, s);
}

}  // namespace bkma
