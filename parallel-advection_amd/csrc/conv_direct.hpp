// The FP64 and FP32 modes of the Conv1d plans (conv_direct.hip).
#pragma once

#include <memory>

#include "stream_scratch.hpp"

namespace bkma {

struct DirectConv {
    bkma_dtype dt = BKMA_F64;
    int B = 0, C = 0, L = 0, K = 0;
    bool mfma = false;       // FP32 matrix cores
    bool lane = false;       // FP64, one output channel per lane
    int ocb = 0, jt = 0;     // channels and columns per thread (matrix form: 16-channel and 16-column blocks per wave;
                             // lane form: lanes across the channels of a group)
    int parts = 1;           // matrix form: waves that share a channel group's columns
    int wpt = 1;             // waves per tile
    int groups = 0;          // channel groups
    int TN = 0, pitch = 0;   // columns per tile, LDS row pitch in elements
    int tiles = 0, total = 0, chunk = 0, owners = 0;
    int slots = 1;           // owners per work-group
    unsigned grid = 0;
    u64 lds_bytes = 0;
    void *w = nullptr;       // packed weights (device, owned by the plan)
    std::unique_ptr<StreamScratch> halo;  // the columns after the owners' chunks, [owners][C][K-1]
};

// The chunk of an owner: tiles [first, end) of the flattened (batch element,
// tile) sequence.
struct ConvChunk {
    int first, end;
    // The first column of batch element b after the chunk, from where on another
    // owner writes the row and a tile takes the copy made before the launch; beyond
    // every column where the chunk goes on past the row.
    __host__ __device__ __forceinline__ int column_after(int b, int tiles, int TN) const {
        const int t = end - b * tiles;
        return t < tiles ? t * TN : 0x7fffffff;
    }
};
__host__ __device__ __forceinline__ ConvChunk conv_chunk(int owner, int chunk, int total) {
    // in 64 bits: total goes up to 2^31 - 1, and an owner past the last one has no tiles
    const i64 first = (i64)owner * chunk, end = first + chunk;
    ConvChunk c;
    c.first = first < total ? (int)first : total;
    c.end = end < total ? (int)end : total;
    return c;
}

// Chooses the launch, allocates and packs the weights on `s`.
bkma_status direct_conv_create(bkma_dtype dt, int B, int C, int L, int K, const void *weight, hipStream_t s,
                               DirectConv *out);
void direct_conv_free(DirectConv &d);
// Runs of one plan may overlap on several streams.
bkma_status direct_conv_run(const DirectConv &d, void *x, const void *bias, hipStream_t s);

}  // namespace bkma
