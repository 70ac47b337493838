// What the attention kernels share: their arguments.
#pragma once
#include "common.hpp"
#include <type_traits>

struct SdpaArgs {
    void *out;
    const half_t *q, *k, *v;
    long qs[4], ks[4], vs[4], os[4];   // (E, L, H, B) element strides
    const void *bias;
    long bs[4];                    // (Lk, Lq, H, B) element strides, 0 = broadcast
    const int *kv_len;
    float *part_o, *part_ml;       // split partials: [split][row][E], [split][row][2] (sdpa_decode_kernel: [row][split])
    unsigned *tickets;             // sdpa_decode_kernel with nsplit > 1: one arrival counter per (head, batch), zero between launches
    // sdpa_decode_kernel only: the newest key/value row (1 x E per head and batch); when set, key kv_len - 1 is
    // taken from here instead of the cache and written into the cache on the way (k, v are then written to)
    const half_t *k_new, *v_new;
    long ns[4];
    int E, Lq, Lk, H, B;
    int out_f32, bias_f32, nsplit;
    float scale;
};

namespace {

constexpr float LOG2E = 1.4426950408889634f;

template <int N, typename F>
__device__ __forceinline__ void static_for(F &&f) {
    if constexpr (N > 0) {
        static_for<N - 1>(f);
        f(std::integral_constant<int, N - 1>{});
    }
}

}  // namespace

// sdpa_tile.hip: 32-query workgroups whose waves share nothing but the final merge, for operands that the fused kernels can address
// and that mi_sdpa_tile_takes.  `f32`: scores and probabilities keep the fp32 that the rows kernel gives them.
constexpr int MI_SDPA_TILE_KEYMASK_MAX = 4096;
bool mi_sdpa_tile_head_size(int64_t E);
bool mi_sdpa_tile_takes(const SdpaArgs &p);
bool mi_sdpa_tile_keymask(const SdpaArgs &p);
int mi_sdpa_tile_launch(const SdpaArgs &p, int waves, bool f32, hipStream_t st);
int mi_sdpa_tile_init();
