// The FP64 and FP32 modes of the Conv1d plans (conv_direct.hip).
#pragma once

#include "common.hpp"

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
    unsigned grid = 0;
    u64 lds_bytes = 0;
    void *w = nullptr;       // packed weights (device, owned by the plan)
    void *halo = nullptr;    // last tiles' neighbour columns, [owners][C][K-1] (device, owned by the plan)
};

// Chooses the launch, allocates and packs the weights on `s`.
bkma_status direct_conv_create(bkma_dtype dt, int B, int C, int L, int K, const void *weight, hipStream_t s,
                               DirectConv *out);
void direct_conv_free(DirectConv &d);
bkma_status direct_conv_run(const DirectConv &d, void *x, const void *bias, hipStream_t s);

}  // namespace bkma
