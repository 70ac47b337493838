// What the attention kernels share: their arguments.
#pragma once
#include "common.hpp"
#include <type_traits>

// The order is the kernels': what flash_tile_kernel reads lies in the first four 64-byte lines.
struct SdpaArgs {
    const half_t *q, *k, *v;
    void *out;
    int Lq, Lk, H, B;
    unsigned div_h, div_x, div_split;      // recip_of(H), of the grid's query blocks (flash_tile_kernel: nqb), of nsplit
    int nqb;                       // flash_tile_kernel: query blocks
    long qs[4], ks[4], vs[4], os[4];   // (E, L, H, B) element strides
    const int *kv_len;
    const void *bias;
    long bs[4];                    // (Lk, Lq, H, B) element strides, 0 = broadcast
    int E, nsplit;
    float scale;
    int out_f32;
    int bias_f32;
    int per;                       // sdpa_decode_kernel: 64-key passes of a split
    // sdpa_decode_kernel only: the newest key/value row (1 x E per head and batch); when set, key kv_len - 1 is
    // taken from here instead of the cache and written into the cache on the way (k, v are then written to)
    const half_t *k_new, *v_new;
    long ns[4];
    unsigned *tickets;             // sdpa_decode_kernel with nsplit > 1: one arrival counter per (head, batch), zero between launches
    float *part_o, *part_ml;       // split partials: [split][row][E], [split][row][2] (sdpa_decode_kernel: [row][split])
};

namespace {

constexpr float LOG2E = 1.4426950408889634f;

// Asks for the argument block at once.  The compiler asks for a field where it is first used, a line of the block at a time and each a trip
// of 200 (replayed graphs) to 700 clocks behind the other; four to six of them stood between these launches and their first load.
// For the decode kernel all of it; for flash_tile_kernel what stands in front of its first load: asking for the rest as well held that load
// back (16 x 8 heads of 256 queries, 72 wide, padded, called from the host: 11.26 us with all of it, 11.05 so), and the strides of
// a mask in a line of their own cost 0.3 us.  The fused kernel lost by any (2 x 16 heads of 300, a mask from query to query: 14.7 | 14.1).
__device__ __forceinline__ void stage_tile_args(const SdpaArgs &p) {
    asm volatile("" ::"s"(p.q), "s"(p.Lq), "s"(p.Lk), "s"(p.H), "s"(p.B), "s"(p.div_h), "s"(p.div_x), "s"(p.nqb), "s"(p.qs[1]), "s"(p.qs[2]), "s"(p.qs[3]), "s"(p.kv_len));
}
__device__ __forceinline__ void stage_decode_args(const SdpaArgs &p) {
    asm volatile("" ::"s"(p.q), "s"(p.k), "s"(p.v), "s"(p.out), "s"(p.Lq), "s"(p.Lk), "s"(p.H), "s"(p.B), "s"(p.div_h), "s"(p.qs[2]), "s"(p.qs[3]),
                 "s"(p.ks[1]), "s"(p.ks[2]), "s"(p.ks[3]), "s"(p.vs[1]), "s"(p.vs[2]), "s"(p.vs[3]), "s"(p.os[2]), "s"(p.os[3]), "s"(p.E),
                 "s"(p.nsplit), "s"(p.scale), "s"(p.kv_len), "s"(p.part_ml), "s"(p.k_new), "s"(p.ns[3]), "s"(p.per));
}

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

// sdpa_decode.hip: one query per (head, batch) in one launch, for operands that 16-byte loads can address.
bool mi_sdpa_decode_takes(const SdpaArgs &p);
int mi_sdpa_decode_splits(int64_t E, int64_t Lk, int64_t H, int64_t B);
int mi_sdpa_decode_launch(const SdpaArgs &p, hipStream_t st);
void mi_sdpa_decode_init();
