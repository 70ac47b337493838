// The arguments the convolution kernels share.
#pragma once
#include "common.hpp"
#include "conv_tile_plan.hpp"

struct ConvArgs : ConvShape {
    const half_t *x, *w, *bias;
    void *out;
};

// conv_tile.hip: the one-launch implicit GEMM over channel-first maps, one group.  Its own estimate, 1e30 where a chunk of one
// channel does not fit the LDS; the launch, MI_DECLINE_EXTENT (nothing enqueued) in that case.
double mi_conv_tile_us(const ConvArgs &a);
int mi_conv_tile(const ConvArgs &a, hipStream_t st);
int mi_conv_tile_init();
