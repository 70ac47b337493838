// What the tiled fp16 GEMM kernels share: their arguments, operand staging, the workgroup -> tile map and the store
// (bias, folded layer norm, activation, residual, clamp, row statistics).
//
// Internal problem statement (row-major):  Y[M x N] = A[M x K] . B  (+ bias)
//   A is K-contiguous.  B is either N-contiguous [K][N] (B_KN) or K-contiguous
//   [N][K].  For a linear layer M = tokens, N = features, A = X, B = W.
#pragma once
#include "common.hpp"
#include <type_traits>

// The order is the kernels': what stands between a launch and its first load lies in the first two 64-byte lines of the
// argument block, what its store needs in the next two (stage_args).
struct GemmArgs {
    const half_t *A, *B;
    long ldA, ldB;
    int M, N, K;
    int NB;                 // columns addressable in B (>= N; a multiple of 8 for the [K][N] layout)
    int tiles_m, tiles_n, group_m;
    unsigned div_width, div_group, div_last;      // tile_of's divisions as multiplications (set_tiles)
    int bias_mode, epi;
    long sA, sB, sY, sBias; // batch strides (elements)
    void *Y;
    long ldY;
    const half_t *bias, *residual;
    long dRes;              // the residual's batch stride is sY + dRes (one position embedding for every image: -sY)
    // Layer norm folded away (mi_lnfold_gemm_f16): A holds the raw rows, B carries gamma, and the store turns an
    // accumulator into r (acc - mu colsum[n]) + biasp[n], with the row's (mu, r) combined from lnf_stats.
    const float *lnf_stats;           // [lnf_nseg][M][2]: (sum, squares about its own mean) of each 32-column segment of a row
    const float *lnf_colsum, *lnf_biasp;      // fp32[N], plane stride lnf_svec
    long lnf_svec;
    int lnf_nseg;
    float lnf_eps;
    // Row statistics of the result for a later folded norm: stats_out[n / 32][m] = (sum, squares about the mean) of the
    // final fp16 values Y[m][32 (n / 32) .. + 32); stats_nseg segments per row.
    float *stats_out;
    int stats_nseg;
    // Tiled kernels and the split-K plane sums: > 0 clamps the fp16 result to [-clamp, clamp] after the residual add,
    // as a separate aten::clamp on Y would (the overflow guard of exported fp16 encoder layers).
    float clamp;
    int out_f32;
    int vec_store;          // Y (and residual) rows allow 16-byte accesses
    ConvGather cv;          // cv.xp != nullptr: B is the im2col matrix of a convolution, gathered on the fly
    NhwcGather ag;          // ag.x != nullptr: A is the patch matrix of a channels-last convolution, gathered on the fly
    // Decode-sized kernels only: the rows of A are layer-normalised over K on their way into LDS
    // (ln_on; gamma, beta may be null), exactly as layernorm_vec_kernel would have written them.
    const half_t *ln_gamma, *ln_beta;
    float ln_eps;
    int ln_on;
    unsigned div_k8;        // recip_of(K / 8)
    // Output side: when lnout is set, the rows of Y are also layer-normalised over N into lnout (dense rows of N
    // halves), as mi_layernorm_f16 on Y would write them (the next block's first norm riding in this GEMM's store).
    half_t *lnout;
    const half_t *lnout_gamma, *lnout_beta;
    float lnout_eps;
    // Measurement only (mi_set_clock_probe): workgroup 0 of a four-wave launch stores {shader clock, 100 MHz clock}
    // here when it starts and again after its last store.  Null in ordinary use.
    unsigned long long *clk;
    // Measurement only (mi_set_phase_probe): every matrix wave of the first phase_wgs workgroups of a four-wave launch
    // stores the shader clocks it spent {before its K loop, in it, issuing its store, waiting for the store to drain}.
    unsigned long long *phase;
    int phase_wgs;
    // Split-K with the partial tiles exchanged between the workgroups of a tile instead of written as planes
    // (gemm_w4_kernel, SK instance): sk_S = 2 workgroups per tile, tiles dealt sk_tpx per XCD; partials in sk_part,
    // per-wave arrival flags in sk_flags (they carry sk_epoch; the last reader of a flag clears it).
    int sk_S, sk_tpx;
    float *sk_part;
    unsigned *sk_flags;
    unsigned sk_epoch;
    int sk_spin;                      // polls before a wave gives up on its partners
    unsigned sk_pub_xor, sk_xcc_xor;  // zero in ordinary use: mi_test_exchange_faults makes the waits fail from the host side
    unsigned *status;                 // the device's sticky status word
};

namespace {

template <int N, typename F>
__device__ __forceinline__ void static_for(F &&f) {
    if constexpr (N > 0) {
        static_for<N - 1>(f);
        f(std::integral_constant<int, N - 1>{});
    }
}

// At the entry of a loader wave, which has asked for nothing.  The branches that part the waves meet again in the compiled code, so that there
// the compiler takes the matrix waves' loads for pending and waits for each where it next writes that register; between direct-to-LDS
// requests, which it does not see, such a wait is one for their data, before the next are asked for.  Here it waits for nothing.
__device__ __forceinline__ void nothing_pending() { __builtin_amdgcn_s_waitcnt(0x0f70); }      // vmcnt(0)

// Kernel arguments come through the scalar cache a 64-byte line at a time: 200 clocks a line in a replayed graph, 550 to 700 where
// the host has just written them, and the compiler asks for a field where it is first used, so that four or five such trips
// stood in a row between a launch and its first load.  Naming the fields at the kernel's first line requests them together.
__device__ __forceinline__ void stage_args(const GemmArgs &p) {
    asm volatile("" ::"s"(p.A), "s"(p.B), "s"(p.ldA), "s"(p.ldB), "s"(p.M), "s"(p.N), "s"(p.K), "s"(p.NB), "s"(p.tiles_m), "s"(p.tiles_n),
                 "s"(p.group_m), "s"(p.div_width), "s"(p.div_group), "s"(p.div_last), "s"(p.bias_mode), "s"(p.epi), "s"(p.sA), "s"(p.sB),
                 "s"(p.Y), "s"(p.ldY), "s"(p.bias), "s"(p.residual), "s"(p.lnf_stats), "s"(p.stats_out), "s"(p.vec_store));
}

// Workgroup id -> output tile.  The hardware deals consecutive workgroups
// round-robin over the 8 XCDs, each with its own L2; this hands every XCD one
// contiguous run of the tile order, and the tile order walks GROUP_M row tiles
// per column tile so a run reuses a small set of A and B panels.
// Its divisions are multiplications by reciprocals the host worked out (set_tiles, divide): three in a row stood between a launch and
// its first load.
__device__ __forceinline__ void tile_of(const GemmArgs &p, int &tm, int &tn) {
    const int pid = blockIdx.x, nwg = p.tiles_m * p.tiles_n;
    const int xcd = pid & 7, idx = pid >> 3;
    const int full = nwg >> 3, rem = nwg & 7;
    const int logical = xcd * full + min(xcd, rem) + idx;
    unsigned in, row;
    const int first = (int)divide(logical, p.group_m * p.tiles_n, p.div_width, in) * p.group_m;
    const int gsz = min(p.tiles_m - first, p.group_m);
    tn = (int)divide(in, gsz, gsz == p.group_m ? p.div_group : p.div_last, row);
    tm = first + (int)row;
}

// The tile grid of a launch.
inline void set_tiles(GemmArgs &a, int bm, int bn) {
    a.tiles_m = (int)ceil_div(a.M, bm);
    a.tiles_n = (int)ceil_div(a.N, bn);
    a.group_m = a.tiles_m < 6 ? a.tiles_m : 6;
    const int last = a.tiles_m % a.group_m;
    a.div_width = recip_of((int64_t)a.group_m * a.tiles_n);
    a.div_group = recip_of(a.group_m);
    a.div_last = recip_of(last ? last : a.group_m);
}

// A folded norm's row statistics, r (acc - mu colsum) + biasp: a row's mean and reciprocal standard deviation over its K elements
// come from the per-segment statistics a producer left (stats[seg][row] = (sum, squares about the segment's own mean)).  One
// pass: the squares between the segments are taken about the first segment's mean, which lies within a segment mean's
// spread of the row mean, so the final subtraction cancels nothing that matters -- sum(x^2) - n mean^2 about zero would.
// r = 1 / sqrt(var + eps), rmu = r * mean.

// Four of colsum's or biasp's floats from n on; past the edge the last ones again (such launches have whole quads of columns and
// whole 64-deep tiles of K).
__device__ __forceinline__ float4v lnf_columns(const GemmArgs &p, const float *vec, int n, long bz) {
    return *reinterpret_cast<const float4v *>(vec + bz * p.lnf_svec + min(n, p.N - 4));
}

// In the matrix waves of a kernel whose K tiles are two segments deep and pass through registers: a lane's rows are those of its
// accumulators, its half of the wave takes every other segment, a load and some eight vector instructions a tile and row, all
// beside the products; what the store needs is in registers under the last tile.  (Requested in the prologue, ten conditional
// loads a lane with a wait where each condition ended, combined in one go ahead of the last tile by four lanes a row and handed
// over through LDS, the norm spilled registers and cost 1370 x 384 -> 1152 2 400 clocks, 11 080 against 8 700 without it;
// now 1 900, of which 1 000 are instructions beside the loop's.  Launch to first product 2 220 -> 2 080, store 2 200 -> 1 790.
// ViT-S of 1370 tokens, 24 such launches: 521 -> 506 us.)
template <int TM>
struct LnfRows {
    const float2v *seg[TM];
    float ref[TM], total[TM], within[TM], between[TM];
    float2v v[2][TM];
    // mw: the wave's first row
    __device__ __forceinline__ LnfRows(const GemmArgs &p, int mw, int lane) {
#pragma unroll
        for (int j = 0; j < TM; j++) {
            seg[j] = reinterpret_cast<const float2v *>(p.lnf_stats) + (long)(lane >> 5) * p.M + min(mw + 32 * j + (lane & 31), p.M - 1);
            total[j] = within[j] = between[j] = 0.0f;
        }
    }
    __device__ __forceinline__ void request(const GemmArgs &p, int set, int kt) {
#pragma unroll
        for (int j = 0; j < TM; j++) v[set][j] = seg[j][(long)(2 * kt) * p.M];
    }
    template <bool FIRST = false>
    __device__ __forceinline__ void take(int set) {
#pragma unroll
        for (int j = 0; j < TM; j++) {
            const float2v s = v[set][j];
            if constexpr (FIRST) {
                float other = s[0];
                ref[j] = s[0];
                swap_rows32(ref[j], other);                       // the first segment's sum, in both halves of the wave
                ref[j] *= 1.0f / 32.0f;
            }
            const float d = fmaf(s[0], 1.0f / 32.0f, -ref[j]);
            total[j] += s[0];
            within[j] += s[1];
            between[j] = fmaf(32.0f * d, d, between[j]);
        }
    }
    __device__ __forceinline__ void finish(const GemmArgs &p, float (&r)[TM], float (&rmu)[TM]) {
        // (a division by K is one by a reciprocal and its remainder, the root of the variance an estimate and a Newton step: as
        // exact to within a last bit, and a third of the instructions between the last statistics and the last product)
        const float k = (float)p.K, ik = __builtin_amdgcn_rcpf(k), inv = fmaf(fmaf(-k, ik, 1.0f), ik, ik);
        auto both = [](float x) { float y = x; swap_rows32(x, y); return x + y; };
        auto over_k = [&](float x) { const float t = x * inv; return fmaf(fmaf(-k, t, x), inv, t); };
#pragma unroll
        for (int j = 0; j < TM; j++) {
            const float mu = over_k(both(total[j])), dm = mu - ref[j];
            const float var = over_k(both(within[j]) + fmaxf(both(between[j]) - k * dm * dm, 0.0f)) + p.lnf_eps;
            const float e = __builtin_amdgcn_rsqf(var);
            r[j] = var > 0.0f ? fmaf(0.5f * e, fmaf(-var * e, e, 1.0f), e) : e;      // (fp16 rows: a variance is 0 or far from the smallest floats)
            rmu[j] = r[j] * mu;
        }
    }
};

// By a wave of its own, beside the K loop of kernels whose tiles go straight to LDS: the matrix waves need (r, r mu) of the
// tile's rows and the tile's columns of colsum and biasp at the store, not before, and in their registers the statistics
// would cost a second workgroup a CU.  (In the prologue they held every wave at the first barrier: 5 000 clocks at 128 rows,
// 10 000 at 192, a trip to memory per batch of loads, then forty dependent steps a row.)  Tile kt covers segments 2 kt and
// 2 kt + 1 (SEGS = 2; a 128-deep tile four): ahead of barrier kt this wave takes in the segments of each of its rows that it
// requested AHEAD tiles earlier, and the result is in the slot when it arrives at the last barrier, which the matrix waves pass
// before they store.  The slot: (r, r mu) of BM rows, BN column sums, BN biases.  LEAD: a barrier comes before tile 0's.
template <int BM, int BN, bool LEAD, int SEGS = 2, typename BarrierF>
__device__ __forceinline__ void lnf_stats_wave(const GemmArgs &p, float2v *slot, int m0, int n0, long bz, int lane, int nk, BarrierF barrier) {
    constexpr int NR = (BM + 63) / 64, AHEAD = 4;
    static_assert((BM % 64 == 0 || BM == 32) && NR * SEGS * AHEAD <= 63, "whole rows per lane; vmcnt is a 6-bit counter");
    constexpr int NC = (BN / 2 + 63) / 64;
    float4v col[NC];
#pragma unroll
    for (int i = 0; i < NC; i++) {
        const int t = min(lane + 64 * i, BN / 2 - 1);
        col[i] = lnf_columns(p, t < BN / 4 ? p.lnf_colsum : p.lnf_biasp, n0 + (t % (BN / 4)) * 4, bz);
    }
    const float2v *seg[NR];
#pragma unroll
    for (int i = 0; i < NR; i++) seg[i] = reinterpret_cast<const float2v *>(p.lnf_stats) + min(m0 + lane + 64 * i, p.M - 1);
    float2v v[AHEAD][NR][SEGS];
    float ref[NR], total[NR], within[NR], between[NR];
#pragma unroll
    for (int i = 0; i < NR; i++) { ref[i] = 0.0f; total[i] = 0.0f; within[i] = 0.0f; between[i] = 0.0f; }
    auto fetch = [&](auto SLOT, int kt) {
        constexpr int sl = decltype(SLOT)::value;
#pragma unroll
        for (int i = 0; i < NR; i++)
#pragma unroll
            for (int h = 0; h < SEGS; h++) v[sl][i][h] = seg[i][(long)min(SEGS * kt + h, p.lnf_nseg - 1) * p.M];
    };
    auto take = [&](auto SLOT, int kt) {
        constexpr int sl = decltype(SLOT)::value;
#pragma unroll
        for (int h = 0; h < SEGS; h++) {
            const int left = p.K - 32 * (SEGS * kt + h);                  // uniform
            if (left <= 0) break;
            const float cnt = left >= 32 ? 32.0f : (float)left, inv = left >= 32 ? 1.0f / 32.0f : 1.0f / (float)left;
#pragma unroll
            for (int i = 0; i < NR; i++) {
                if (kt == 0 && h == 0) ref[i] = v[sl][i][0][0] * inv;
                const float d = fmaf(v[sl][i][h][0], inv, -ref[i]);
                total[i] += v[sl][i][h][0];
                within[i] += v[sl][i][h][1];
                between[i] = fmaf(cnt * d, d, between[i]);
            }
        }
    };
    // tiles 0 .. AHEAD - 1 are requested at once; tile kt + AHEAD right after tile kt is taken in
    static_for<AHEAD>([&](auto S) { if (decltype(S)::value < nk) fetch(S, decltype(S)::value); });
    if (LEAD) barrier();
#pragma unroll
    for (int i = 0; i < NC; i++) {
        const int t = lane + 64 * i;
        if (t < BN / 2) *reinterpret_cast<float4v *>(reinterpret_cast<float *>(slot + BM) + t / (BN / 4) * BN + (t % (BN / 4)) * 4) = col[i];
    }
    for (int kt0 = 0; kt0 < nk; kt0 += AHEAD) {
        static_for<AHEAD>([&](auto S) {
            const int kt = kt0 + decltype(S)::value;
            if (kt < nk) {
                // requests complete in order: what was requested after tile kt may still be on its way
                if (kt + AHEAD - 1 < nk) asm volatile("s_waitcnt vmcnt(%0)" ::"n"((AHEAD - 1) * NR * SEGS) : "memory");
                else asm volatile("s_waitcnt vmcnt(0)" ::: "memory");
                take(S, kt);
                if (kt + AHEAD < nk) fetch(S, kt + AHEAD);
                if (kt + 1 == nk) {
#pragma unroll
                    for (int i = 0; i < NR; i++) {
                        const float mu = total[i] / (float)p.K, dm = mu - ref[i];
                        const float m2 = within[i] + fmaxf(between[i] - (float)p.K * dm * dm, 0.0f);
                        const float r = 1.0f / sqrtf(m2 / (float)p.K + p.lnf_eps);
                        const float2v o = {r, r * mu};
                        if (BM % 64 == 0 || lane < BM) slot[lane + 64 * i] = o;
                    }
                    asm volatile("s_waitcnt lgkmcnt(0)" ::: "memory");
                }
                barrier();                                      // B_kt
            }
        });
    }
}

// ------------------------------------------------------------------------------------------
// Accumulator tile -> memory, shared by the tiled kernels.
// acc[i][j][r]: n = n0 + wn*WTN + 32 i + 8 (r/4) + 4 (lane/32) + r%4,  m = m0 + wm*WTM + 32 j + lane%32.
// Each wave stages one 32 x WTN sub-tile at a time in its own LDS region (bias
// joined in fp32, one rounding), then reads it back row-wise so that the
// activation, the residual add and the global stores run on 16-byte vectors
// that are contiguous along the output row.  The caller has synchronised the
// workgroup after its last read of the operand tiles.
// The column bias of a wave's sub-tile, in the accumulator's order: cb[i][g] covers
// n = n0 + wn*WTN + 32 i + 8 g + 4 (lane/32) .. +3.  Fetched by the kernels ahead of their last
// k-step so that the epilogue does not start with a trip to memory; the choices are uniform, no load stands behind a condition
// of its lane.  Four columns are one load at any address, moved back to end at N where they would pass it: a width off four then has
// the quad that N ends in shifted, which settle_col_bias undoes where the bias is used.
template <int TN, int WTN>
__device__ __forceinline__ void load_col_bias(const GemmArgs &p, half4v (&cb)[TN][4], int n0, int wn, int lane, long bz) {
    const half4v z = {(half_t)0.0f, (half_t)0.0f, (half_t)0.0f, (half_t)0.0f};
    const int nl = n0 + wn * WTN + 4 * (lane >> 5);
    if (p.bias_mode != MI_BIAS_COL) {
#pragma unroll
        for (int i = 0; i < TN; i++)
#pragma unroll
            for (int g = 0; g < 4; g++) cb[i][g] = z;
        return;
    }
    const half_t *bias = p.bias + bz * p.sBias;
    if (p.N >= 4) {
#pragma unroll
        for (int i = 0; i < TN; i++)
#pragma unroll
            for (int g = 0; g < 4; g++) __builtin_memcpy(&cb[i][g], bias + min(nl + 32 * i + 8 * g, p.N - 4), 8);
    } else {
#pragma unroll
        for (int i = 0; i < TN; i++)
#pragma unroll
            for (int g = 0; g < 4; g++)
#pragma unroll
                for (int e = 0; e < 4; e++) cb[i][g][e] = bias[min(nl + 32 * i + 8 * g + e, p.N - 1)];
    }
}
// nw: the wave's first column.  Only a wave that N ends in has such a quad; quads past N reach nothing.
template <int TN, int WTN>
__device__ __forceinline__ void settle_col_bias(const GemmArgs &p, half4v (&cb)[TN][4], int nw, int lane) {
    if (p.N % 4 == 0 || p.N < 4 || nw + WTN <= p.N) return;       // uniform
#pragma unroll
    for (int i = 0; i < TN; i++)
#pragma unroll
        for (int g = 0; g < 4; g++) {
            const int back = min(max(nw + 32 * i + 8 * g + 4 * (lane >> 5) + 4 - p.N, 0), 3);
            cb[i][g] = __builtin_bit_cast(half4v, __builtin_bit_cast(uint64_t, cb[i][g]) >> (16 * back));
        }
}

// What the store of a folded layer norm carries (by value, so that it stays in registers): (r, r mu) of the lane's rows
// m0 + wm WTM + 32 j + lane % 32, and the LDS copy of the tile's colsum (bn floats) followed by its biasp.
template <int TM>
struct LnFold {
    bool on = false;
    float r[TM] = {}, rmu[TM] = {};
    const float *col = nullptr;
    int bn = 0;
    // columns 32 i + 8 g + 4 (lane / 32) .. +3 of the wave's sub-tile, which starts at column `wcol` of the tile
    __device__ __forceinline__ float4v colsum(int i, int g, int wcol, int hl) const { return *reinterpret_cast<const float4v *>(col + wcol + 32 * i + 8 * g + 4 * hl); }
    __device__ __forceinline__ float4v biasp(int i, int g, int wcol, int hl) const { return *reinterpret_cast<const float4v *>(col + bn + wcol + 32 * i + 8 * g + 4 * hl); }
};
// The same with the columns in registers, fetched ahead of the last tile like the column bias.
template <int TM, int TN>
struct LnFoldRegs {
    static constexpr bool on = true;
    float r[TM], rmu[TM];
    float4v c[TN][4], b[TN][4];
    // nw: the wave's first column
    __device__ __forceinline__ void load(const GemmArgs &p, int nw, int lane, long bz) {
#pragma unroll
        for (int i = 0; i < TN; i++)
#pragma unroll
            for (int g = 0; g < 4; g++) {
                const int n = nw + 32 * i + 8 * g + 4 * (lane >> 5);
                c[i][g] = lnf_columns(p, p.lnf_colsum, n, bz);
                b[i][g] = lnf_columns(p, p.lnf_biasp, n, bz);
            }
    }
    __device__ __forceinline__ float4v colsum(int i, int g, int, int) const { return c[i][g]; }
    __device__ __forceinline__ float4v biasp(int i, int g, int, int) const { return b[i][g]; }
};
template <int EPI, int TM, int TN, int WTM, int WTN, int NWAVES, int LDS_BYTES, typename LN>
__device__ __forceinline__ void store_tile_epi(const GemmArgs &p, float16v (&acc)[TN][TM], const half4v (&loaded)[TN][4], char *smem, int m0, int n0, int wm, int wn,
                                               int wave, int lane, long bz, const LN &ln) {
    const int frow = lane & 31;
    const half_t *bias = p.bias ? p.bias + bz * p.sBias : nullptr;
    constexpr int SLD_H = WTN + 8;                 // halves per staged row (fp16 output)
    constexpr int SLD_F = WTN + 4;                 // floats per staged row (fp32 output)
    constexpr int STAGE_BYTES = 32 * SLD_F * 4;
    static_assert(STAGE_BYTES * NWAVES <= LDS_BYTES, "epilogue staging exceeds the operand LDS");
    char *stage = smem + wave * STAGE_BYTES;
    const int hl = lane >> 5;
    half4v cb[TN][4];
#pragma unroll
    for (int i = 0; i < TN; i++)
#pragma unroll
        for (int g = 0; g < 4; g++) cb[i][g] = loaded[i][g];
    settle_col_bias<TN, WTN>(p, cb, n0 + wn * WTN, lane);
    // Row biases for all of the wave's rows before the first store (store_tile_simple says why).
    float brow_j[TM];
#pragma unroll
    for (int j = 0; j < TM; j++) {
        const int m = m0 + wm * WTM + 32 * j + frow;
        brow_j[j] = (p.bias_mode == MI_BIAS_ROW && m < p.M) ? (float)bias[m] : 0.0f;
    }
    static_for<TM>([&](auto J) {
        constexpr int j = decltype(J)::value;
        const int mrow = m0 + wm * WTM + 32 * j;
        const float brow = brow_j[j];
#pragma unroll
        for (int i = 0; i < TN; i++) {
            // folded layer norm: this lane's columns of colsum and biasp from their LDS copy, a 32-column group at a time
            float4v lc4[4], lb4[4];
            if (ln.on) {
#pragma unroll
                for (int g = 0; g < 4; g++) { lc4[g] = ln.colsum(i, g, wn * WTN, hl); lb4[g] = ln.biasp(i, g, wn * WTN, hl); }
            }
#pragma unroll
            for (int g = 0; g < 4; g++) {
                const int nl = 32 * i + 8 * g + 4 * hl;
                const int n = n0 + wn * WTN + nl;
                float v[4];
                if (ln.on) {      // uniform: r (acc - mu colsum) + biasp
#pragma unroll
                    for (int e = 0; e < 4; e++) v[e] = fmaf(acc[i][j][4 * g + e], ln.r[j], fmaf(-ln.rmu[j], lc4[g][e], lb4[g][e]));
                } else {
#pragma unroll
                    for (int e = 0; e < 4; e++) v[e] = acc[i][j][4 * g + e] + brow + (float)cb[i][g][e];
                }
                if (p.out_f32) {
                    float4v o = {v[0], v[1], v[2], v[3]};
                    *reinterpret_cast<float4v *>(reinterpret_cast<float *>(stage) + frow * SLD_F + nl) = o;
                } else {
                    half4v o = {(half_t)v[0], (half_t)v[1], (half_t)v[2], (half_t)v[3]};
                    *reinterpret_cast<half4v *>(reinterpret_cast<half_t *>(stage) + frow * SLD_H + nl) = o;
                }
            }
        }
        // A wave reads back only what it staged itself, and its LDS operations complete in order:
        // no workgroup barrier, only a stop for the compiler.
        asm volatile("s_waitcnt lgkmcnt(0)" ::: "memory");
        if (p.out_f32) {
            constexpr int CPR = WTN / 4;
            for (int c = lane; c < 32 * CPR; c += 64) {
                const int row = c / CPR, ch = c % CPR;
                const int m = mrow + row, n = n0 + wn * WTN + ch * 4;
                if (m < p.M && n < p.N) {
                    float4v x = *reinterpret_cast<const float4v *>(reinterpret_cast<const float *>(stage) + row * SLD_F + ch * 4);
                    float *yp = reinterpret_cast<float *>(p.Y) + bz * p.sY + (long)m * p.ldY + n;
#pragma unroll
                    for (int e = 0; e < 4; e++) x[e] = apply_epi_c<EPI>(x[e]);
                    if (n + 3 < p.N) __builtin_memcpy(yp, &x, 16);      // one 16-byte store at any address
                    else for (int e = 0; e < 4; e++) if (n + e < p.N) yp[e] = x[e];
                }
            }
        } else {
            constexpr int CPR = WTN / 8;
            static_assert((32 * CPR) % 64 == 0 && CPR % 4 == 0, "whole waves walk the staged tile; four lanes hold a 32-column segment");
            for (int c = lane; c < 32 * CPR; c += 64) {
                const int row = c / CPR, ch = c % CPR;
                const int m = mrow + row, n = n0 + wn * WTN + ch * 8;
                half8v x = {};
                if (m < p.M && n < p.N) {
                    x = *reinterpret_cast<const half8v *>(reinterpret_cast<const half_t *>(stage) + row * SLD_H + ch * 8);
                    const long off = bz * p.sY + (long)m * p.ldY + n;
                    half_t *yp = reinterpret_cast<half_t *>(p.Y) + off;
                    x = apply_epi8<EPI>(x);
                    if (n + 7 < p.N) {
                        if (p.residual) {
                            half8v rv;
                            __builtin_memcpy(&rv, p.residual + off + bz * p.dRes, 16);
#pragma unroll
                            for (int e = 0; e < 8; e++) x[e] = (half_t)((float)x[e] + (float)rv[e]);
                        }
                        if (p.clamp > 0.0f) {
#pragma unroll
                            for (int e = 0; e < 8; e++) x[e] = (half_t)fminf(fmaxf((float)x[e], -p.clamp), p.clamp);
                        }
                        __builtin_memcpy(yp, &x, 16);
                    } else {
                        for (int e = 0; e < 8; e++) {
                            if (n + e < p.N) {
                                half_t o = x[e];
                                if (p.residual) o = (half_t)((float)o + (float)p.residual[off + bz * p.dRes + e]);
                                if (p.clamp > 0.0f) o = (half_t)fminf(fmaxf((float)o, -p.clamp), p.clamp);
                                yp[e] = o;
                            }
                        }
                    }
                }
                if (p.stats_out) {      // uniform; the launcher admits it with 16-byte stores and N % 8 == 0 only
                    // the four lanes of a quad hold the 32 columns of one segment of one row (chunks that lie past N
                    // or below M count nothing): sum, then squares about the segment's own mean, both over the quad
                    const bool have = m < p.M && n < p.N;
                    float cnt = have ? 8.0f : 0.0f, sum = 0.0f;
#pragma unroll
                    for (int e = 0; e < 8; e++) sum += have ? (float)x[e] : 0.0f;
                    sum += lane_xor<1>(sum); sum += lane_xor<2>(sum);
                    cnt += lane_xor<1>(cnt); cnt += lane_xor<2>(cnt);
                    const float mean = sum / fmaxf(cnt, 1.0f);
                    float sq = 0.0f;
#pragma unroll
                    for (int e = 0; e < 8; e++) { const float d = (float)x[e] - mean; sq = have ? fmaf(d, d, sq) : sq; }
                    sq += lane_xor<1>(sq); sq += lane_xor<2>(sq);
                    if (have && (ch & 3) == 0) {
                        const float2v o = {sum, sq};
                        *reinterpret_cast<float2v *>(p.stats_out + ((long)(n / 32) * p.M + m) * 2) = o;
                    }
                }
            }
        }
        asm volatile("s_waitcnt lgkmcnt(0)" ::: "memory");
    });
}

// Block j (32 rows) of a wave's accumulators -> its staging area `dst` (32 rows of WTN + 8 halves), rounded to fp16 once
// with the column bias -- or the folded layer norm's r (acc - mu colsum) + biasp -- joined in fp32.
template <int j, int TM, int TN, int WTN, typename LN>
__device__ __forceinline__ void stage_block(float16v (&acc)[TN][TM], const half4v (&cb)[TN][4], const LN &ln, int wn, char *dst, int lane) {
    constexpr int SLD_H = WTN + 8;
    const int frow = lane & 31, hl = lane >> 5;
    half_t *st = reinterpret_cast<half_t *>(dst) + frow * SLD_H + 4 * hl;
#pragma unroll
    for (int i = 0; i < TN; i++)
#pragma unroll
        for (int g = 0; g < 4; g++) {
            const int nl = 32 * i + 8 * g;
            float v[4];
            if (ln.on) {      // uniform
                const float4v lc = ln.colsum(i, g, wn * WTN, hl), lb = ln.biasp(i, g, wn * WTN, hl);
#pragma unroll
                for (int e = 0; e < 4; e++) v[e] = fmaf(acc[i][j][4 * g + e], ln.r[j], fmaf(-ln.rmu[j], lc[e], lb[e]));
            } else {
#pragma unroll
                for (int e = 0; e < 4; e++) v[e] = acc[i][j][4 * g + e] + (float)cb[i][g][e];
            }
            const half4v o = {(half_t)v[0], (half_t)v[1], (half_t)v[2], (half_t)v[3]};
            *reinterpret_cast<half4v *>(st + nl) = o;
        }
}

// The common store: fp16 output in whole 16-byte chunks, column bias (or a folded layer norm), optional activation,
// residual, clamp and row statistics; no row bias, no fp32 output, no ragged N.
//
// Loads and stores of a wave share one counter and complete in order, so a wait for a load -- wherever the compiler
// places it -- is also a wait for every store issued before that load to be acknowledged: a trip of two microseconds
// under the burst of all workgroups' stores.  The general store above pays it once per 32-row block of a wave's tile
// and once per residual chunk (8 000 clocks of a 44 000-clock launch at 1500 x 1280 -> 5120).  Here nothing is fetched
// behind a store that anybody then waits for: the caller's column bias is pinned in registers ahead of the first store,
// and the residual chunks of block j + 1 are requested before block j's stores go out.
// Same arithmetic as the general store (bias joined in fp32, one rounding, activation on the rounded value, residual,
// clamp), so the two give the same bits.  Two staging areas a wave: block j + 1 is staged while block j's chunks are on
// their way back from the LDS (a wave's LDS operations complete in order: no wait between staging a block and reading it).
__device__ __forceinline__ bool store_is_simple(const GemmArgs &p) { return !p.out_f32 && p.vec_store && p.N % 8 == 0 && p.bias_mode != MI_BIAS_ROW; }

// A wave's residual chunks of its first 32-row block, which the common store can be handed instead of fetching them itself: a kernel
// that asks for them while its products run spares the store a trip to memory.
template <int WTN>
struct ResidualAhead {
    static constexpr int CPR = WTN / 8, RPI = 64 / CPR, NIT = 32 / RPI;
    half8v v[NIT];
    // (mw, nw): the wave's first row and column
    __device__ __forceinline__ void request(const GemmArgs &p, int mw, int nw, int lane, long bz) {
        const int ch = lane % CPR, r0 = lane / CPR, n = nw + ch * 8;
        if (!p.residual || !store_is_simple(p)) {                 // uniform
#pragma unroll
            for (int t = 0; t < NIT; t++) v[t] = half8v{};
            return;
        }
        const half_t *const base = p.residual + bz * (p.sY + p.dRes) + min(n, p.N - 8);      // rows and columns past the edge: the last ones
#pragma unroll
        for (int t = 0; t < NIT; t++) v[t] = as_half8(ldg16(base + (long)min(mw + r0 + t * RPI, p.M - 1) * p.ldY));
    }
};

template <int EPI, int TM, int TN, int WTM, int WTN, int NWAVES, int LDS_BYTES, typename LN>
__device__ __forceinline__ void store_tile_simple(const GemmArgs &p, float16v (&acc)[TN][TM], const half4v (&cb)[TN][4], char *smem, int m0, int n0, int wm, int wn,
                                                  int wave, int lane, long bz, const LN &ln, const ResidualAhead<WTN> *ahead) {
    constexpr int SLD_H = WTN + 8, BUF_BYTES = 32 * SLD_H * 2;      // halves per staged row; one staging area
    constexpr int CPR = WTN / 8, RPI = 64 / CPR, NIT = 32 / RPI;     // 16-byte chunks per row; rows a wave covers at a time; chunks per lane and block
    static_assert(2 * BUF_BYTES * NWAVES <= LDS_BYTES && 64 % CPR == 0 && CPR % 4 == 0, "two staging areas a wave; four lanes hold a 32-column segment");
    char *const buf = smem + wave * 2 * BUF_BYTES;
    const int frow = lane & 31, hl = lane >> 5;
    const int ch = lane % CPR, r0 = lane / CPR;                      // this lane's chunks of a block: rows r0 + RPI t, columns 8 ch ..
    const int mw = m0 + wm * WTM, n = n0 + wn * WTN + ch * 8;
    const bool col_ok = n < p.N;                                     // N % 8 == 0: a chunk that starts below N ends below it
    const long off0 = bz * p.sY + (long)(mw + r0) * p.ldY + n;
    half_t *const ybase = reinterpret_cast<half_t *>(p.Y) + off0;
    const half_t *const rbase = p.residual ? p.residual + bz * (p.sY + p.dRes) + min(n, p.N - 8) : nullptr;
#pragma unroll
    for (int i = 0; i < TN; i++)
#pragma unroll
        for (int g = 0; g < 4; g++) asm volatile("" ::"v"(cb[i][g]));
    auto stage = [&](auto J) {
        constexpr int j = decltype(J)::value;
        stage_block<j, TM, TN, WTN>(acc, cb, ln, wn, buf + (j & 1) * BUF_BYTES, lane);
    };
    half8v res[2][NIT];
    auto fetch_residual = [&](auto J) {
        constexpr int j = decltype(J)::value;
#pragma unroll
        for (int t = 0; t < NIT; t++) res[j & 1][t] = as_half8(ldg16(rbase + (long)min(mw + 32 * j + r0 + t * RPI, p.M - 1) * p.ldY));
    };
    if (rbase) {
        if (ahead) {
#pragma unroll
            for (int t = 0; t < NIT; t++) res[0][t] = ahead->v[t];
        } else fetch_residual(std::integral_constant<int, 0>{});
    }
    stage(std::integral_constant<int, 0>{});
    static_for<TM>([&](auto J) {
        constexpr int j = decltype(J)::value;
        const half_t *rd = reinterpret_cast<const half_t *>(buf + (j & 1) * BUF_BYTES) + r0 * SLD_H + ch * 8;
        half8v x[NIT];
#pragma unroll
        for (int t = 0; t < NIT; t++) x[t] = *reinterpret_cast<const half8v *>(rd + t * RPI * SLD_H);
        if constexpr (j + 1 < TM) {
            stage(std::integral_constant<int, j + 1>{});
            if (rbase) fetch_residual(std::integral_constant<int, j + 1>{});
        }
#pragma unroll
        for (int t = 0; t < NIT; t++) {
            const int m = mw + 32 * j + r0 + t * RPI;
            const bool have = col_ok && m < p.M;
            x[t] = apply_epi8<EPI>(x[t]);
            if (rbase) {
#pragma unroll
                for (int e = 0; e < 8; e++) x[t][e] = (half_t)((float)x[t][e] + (float)res[j & 1][t][e]);
            }
            if (p.clamp > 0.0f) {
#pragma unroll
                for (int e = 0; e < 8; e++) x[t][e] = (half_t)fminf(fmaxf((float)x[t][e], -p.clamp), p.clamp);
            }
            if (have) *reinterpret_cast<half8v *>(ybase + (long)(32 * j + t * RPI) * p.ldY) = x[t];
            if (p.stats_out) {      // uniform
                // the four lanes of a quad hold the 32 columns of one segment of one row (chunks that lie past N or
                // below M count nothing): sum, then squares about the segment's own mean, both over the quad
                float cnt = have ? 8.0f : 0.0f, sum = 0.0f;
#pragma unroll
                for (int e = 0; e < 8; e++) sum += have ? (float)x[t][e] : 0.0f;
                sum += lane_xor<1>(sum); sum += lane_xor<2>(sum);
                cnt += lane_xor<1>(cnt); cnt += lane_xor<2>(cnt);
                const float mean = sum / fmaxf(cnt, 1.0f);
                float sq = 0.0f;
#pragma unroll
                for (int e = 0; e < 8; e++) { const float d = (float)x[t][e] - mean; sq = have ? fmaf(d, d, sq) : sq; }
                sq += lane_xor<1>(sq); sq += lane_xor<2>(sq);
                if (have && (ch & 3) == 0) {
                    const float2v o = {sum, sq};
                    *reinterpret_cast<float2v *>(p.stats_out + ((long)(n / 32) * p.M + m) * 2) = o;
                }
            }
        }
    });
}

// The four-wave kernel's store, shared between a matrix wave and the helper wave on its SIMD.  One wave issues a vector
// instruction every eight clocks, a SIMD takes one every four: the erf-GELU of a 128 x 256 tile (a reciprocal, an
// exponential and then thirteen other vector instructions on each of 128 values a lane) cost a lone matrix wave 14 600
// clocks, 8 100 with a helper (apply_epi8 has fewer now), and the plain store gains too (1500 x 1280 -> 5120 + bias: 21.8 us against 22.8).  The
// matrix wave stages its 32-row blocks as in store_tile_simple and takes the first half of each block's chunks, the
// helper the second half; a workgroup barrier per block says "block j is staged" (a wave passes barrier j + 1 only
// when it has block j's chunks in registers, so staging block j + 2 over block j's area after that barrier is safe).
// Launches without residual, clamp or statistics only: the others keep store_tile_simple on the matrix waves alone.
__host__ __device__ __forceinline__ bool coop_store_applies(const GemmArgs &p) {
    return !p.out_f32 && p.vec_store && p.N % 8 == 0 && p.bias_mode != MI_BIAS_ROW && !p.residual && !(p.clamp > 0.0f) && !p.stats_out;
}
template <int EPI, int TM, int WTN, bool HELPER, typename StageF, typename BarrierF>
__device__ __forceinline__ void store_coop_epi(const GemmArgs &p, char *buf, int mw, int nw, int lane, long bz, StageF stage, BarrierF barrier) {
    constexpr int SLD_H = WTN + 8, BUF_BYTES = 32 * SLD_H * 2;
    constexpr int CPR = WTN / 8, RPI = 64 / CPR, NIT = 32 / RPI, T0 = HELPER ? NIT / 2 : 0, T1 = HELPER ? NIT : NIT / 2;
    static_assert(NIT % 2 == 0, "the chunks of a block split in two");
    const int ch = lane % CPR, r0 = lane / CPR;
    const int n = nw + ch * 8;
    const bool col_ok = n < p.N;
    half_t *const ybase = reinterpret_cast<half_t *>(p.Y) + bz * p.sY + (long)(mw + r0) * p.ldY + n;
    if constexpr (!HELPER) stage(std::integral_constant<int, 0>{});
    static_for<TM>([&](auto J) {
        constexpr int j = decltype(J)::value;
        barrier();                                             // block j is staged
        const half_t *rd = reinterpret_cast<const half_t *>(buf + (j & 1) * BUF_BYTES) + r0 * SLD_H + ch * 8;
        half8v x[T1 - T0];
#pragma unroll
        for (int t = T0; t < T1; t++) x[t - T0] = *reinterpret_cast<const half8v *>(rd + t * RPI * SLD_H);
        if constexpr (!HELPER && j + 1 < TM) stage(std::integral_constant<int, j + 1>{});
#pragma unroll
        for (int t = T0; t < T1; t++) {
            x[t - T0] = apply_epi8<EPI>(x[t - T0]);
            if (col_ok && mw + 32 * j + r0 + t * RPI < p.M) *reinterpret_cast<half8v *>(ybase + (long)(32 * j + t * RPI) * p.ldY) = x[t - T0];
        }
    });
}
template <int TM, int WTN, bool HELPER, typename StageF, typename BarrierF>
__device__ __forceinline__ void store_coop(const GemmArgs &p, char *buf, int mw, int nw, int lane, long bz, StageF stage, BarrierF barrier) {
    switch (p.epi) {
    case MI_EPI_GELU_ERF: store_coop_epi<MI_EPI_GELU_ERF, TM, WTN, HELPER>(p, buf, mw, nw, lane, bz, stage, barrier); break;
    case MI_EPI_GELU_TANH: store_coop_epi<MI_EPI_GELU_TANH, TM, WTN, HELPER>(p, buf, mw, nw, lane, bz, stage, barrier); break;
    case MI_EPI_RELU: store_coop_epi<MI_EPI_RELU, TM, WTN, HELPER>(p, buf, mw, nw, lane, bz, stage, barrier); break;
    default: store_coop_epi<MI_EPI_NONE, TM, WTN, HELPER>(p, buf, mw, nw, lane, bz, stage, barrier); break;
    }
}

// The activation is a compile-time choice inside the store loops: one uniform branch per tile
// instead of one per element.
template <int TM, int TN, int WTM, int WTN, int NWAVES, int LDS_BYTES, typename LN = LnFold<TM>>
__device__ __forceinline__ void store_tile(const GemmArgs &p, float16v (&acc)[TN][TM], const half4v (&cb)[TN][4], char *smem, int m0, int n0, int wm, int wn,
                                           int wave, int lane, long bz, const LN &ln = LN{}, const ResidualAhead<WTN> *ahead = nullptr) {
    if (store_is_simple(p)) {
        switch (p.epi) {
        case MI_EPI_GELU_ERF: store_tile_simple<MI_EPI_GELU_ERF, TM, TN, WTM, WTN, NWAVES, LDS_BYTES>(p, acc, cb, smem, m0, n0, wm, wn, wave, lane, bz, ln, ahead); break;
        case MI_EPI_GELU_TANH: store_tile_simple<MI_EPI_GELU_TANH, TM, TN, WTM, WTN, NWAVES, LDS_BYTES>(p, acc, cb, smem, m0, n0, wm, wn, wave, lane, bz, ln, ahead); break;
        case MI_EPI_RELU: store_tile_simple<MI_EPI_RELU, TM, TN, WTM, WTN, NWAVES, LDS_BYTES>(p, acc, cb, smem, m0, n0, wm, wn, wave, lane, bz, ln, ahead); break;
        default: store_tile_simple<MI_EPI_NONE, TM, TN, WTM, WTN, NWAVES, LDS_BYTES>(p, acc, cb, smem, m0, n0, wm, wn, wave, lane, bz, ln, ahead); break;
        }
        return;
    }
    switch (p.epi) {
    case MI_EPI_GELU_ERF: store_tile_epi<MI_EPI_GELU_ERF, TM, TN, WTM, WTN, NWAVES, LDS_BYTES>(p, acc, cb, smem, m0, n0, wm, wn, wave, lane, bz, ln); break;
    case MI_EPI_GELU_TANH: store_tile_epi<MI_EPI_GELU_TANH, TM, TN, WTM, WTN, NWAVES, LDS_BYTES>(p, acc, cb, smem, m0, n0, wm, wn, wave, lane, bz, ln); break;
    case MI_EPI_RELU: store_tile_epi<MI_EPI_RELU, TM, TN, WTM, WTN, NWAVES, LDS_BYTES>(p, acc, cb, smem, m0, n0, wm, wn, wave, lane, bz, ln); break;
    default: store_tile_epi<MI_EPI_NONE, TM, TN, WTM, WTN, NWAVES, LDS_BYTES>(p, acc, cb, smem, m0, n0, wm, wn, wave, lane, bz, ln); break;
    }
}

template <typename KernelT>
int raise_lds(KernelT kern, int bytes) {
    return hipFuncSetAttribute(reinterpret_cast<const void *>(kern), hipFuncAttributeMaxDynamicSharedMemorySize, bytes) == hipSuccess ? 0 : 1;
}

template <int BM, int BN, int BK>
constexpr int gemm_lds_bytes() {
    constexpr int kc = BN * (BK + 8), kn = BK * (BN + 32);       // B buffer in either layout
    return 2 * (BM * (BK + 8) + (kc > kn ? kc : kn)) * 2;
}

// Y (and residual) rows allow 16-byte accesses
bool rows_vec16(const GemmArgs &a) {
    return a.out_f32 ? (a.ldY % 4 == 0 && a.sY % 4 == 0 && aligned_to(a.Y, 16))
                     : (a.ldY % 8 == 0 && a.sY % 8 == 0 && aligned_to(a.Y, 16) && (!a.residual || aligned_to(a.residual, 16)));
}

}  // namespace

// gemm_skinny.hip: decode-sized calls.
constexpr size_t SKINNY_FK_LDS_MAX = 128 * 1024;    // activations of the [F][K] decode-sized kernels: M rows of K halves
// Up to eight rows; `ws`: the fp32 planes of mi_skinny_splits K-slices ([K][F] weights only).
int mi_skinny_launch(const GemmArgs &a, bool b_kn, void *ws, size_t ws_bytes, hipStream_t st);
int mi_skinny_splits(int64_t K, int64_t F);
int mi_skinny_slices(int64_t T, int64_t K, int64_t F, int64_t ldA, int64_t ldB);      // those that run: one where the call goes to 32 x 32 tiles
double mi_deep_us(int64_t T, int64_t K, int64_t F);      // gemm.hip's estimate of gemm_deep_kernel, at most one workgroup a CU; infinite otherwise
int mi_skinny_init();
// gemm_pipe.hip: the register-staged pipelined kernel.  `tile` indexes TILE_MODELS (gemm.hip).
int mi_pipe_launch(int tile, const GemmArgs &a, bool b_kn, int64_t nbatch, hipStream_t st);
int mi_pipe_launch_ln(bool wide, const GemmArgs &a, bool b_kn, hipStream_t st);
int mi_pipe_init();
// gemm_ring.hip: small grids of ordinary operands, and patch matrices of a convolution.
int mi_ring_launch(const GemmArgs &a, bool b_kn, int64_t nbatch, hipStream_t st);
int mi_ring_init();
// gemm_deep.hip: few output tiles, of ordinary operands (split_k: K over its waves) and of patch matrices (always).
bool mi_deep_takes(int64_t ldA, int64_t ldB);      // the pitches of ordinary operands
int mi_deep_launch(const GemmArgs &a, bool split_k, bool b_kn, int64_t nbatch, hipStream_t st);
int mi_deep_init();
// gemm_any.hip: the kernels for operands and extents that the others do not take.
int mi_any_launch(const GemmArgs &a, bool b_kn, bool addressable, int64_t nbatch, hipStream_t st);
int mi_any_init();
