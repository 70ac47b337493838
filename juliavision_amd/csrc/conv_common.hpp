// The arguments the convolution kernels share.
#pragma once
#include "common.hpp"
#include "conv_tile_plan.hpp"

struct ConvArgs : ConvShape {
    const half_t *x, *w, *bias;
    void *out;
};

// conv_tile.hip: the one-launch implicit GEMM over channel-first maps, one group.  MI_DECLINE_EXTENT (nothing enqueued)
// where its own estimate is not below limit_us, or where a chunk of one channel does not fit the LDS.
int mi_conv_tile(const ConvArgs &a, double limit_us, hipStream_t st);
int mi_conv_tile_init();
