// fp16 GEMM for gfx950, 32 x 32 tiles, the waves of a long K splitting it: grids of few output tiles, of ordinary operands and of
// convolutions' patch matrices.
#include "gemm_common.hpp"

// Sixteen zero bytes for loads of chunks past the end of K.
static __device__ __align__(16) unsigned deep_zero_words[4];

namespace {

// A workgroup owns a 32 x 32 tile.  Two loader waves keep a ring of 128-deep stages filled (gemm_ring_kernel says how).  NW = 4: each of
// four matrix waves holds all of the tile in accumulators and takes two of the eight 16-deep steps of every stage; the partial tiles
// meet in LDS and wave 0 stores the sum, eight chains of fp32 sums an element (sixteen past K = 4096), added pairwise.  NW = 1, for a short K: one wave
// takes all steps in one chain, the other tiles' order and bits.
//
// What bounds a small grid is its CUs' vector-memory paths: a 64 x 64 tile takes 256 clocks of loads per 64 k, and 24 of them (70 x
// 3072 -> 768) leave the paths of the other CUs idle.  A quarter of the tile is half of the bytes a CU on four times the CUs; K split
// over the waves reads every fragment once, 16 KB of LDS traffic in and 16 out a stage.  Against the 64 x 64 ring or the K-split
// planes taken before, in us: 70 x 3072 -> 768 11.5 -> 6.9 ([N][K]), 11.0 -> 8.8 ([K][N]: 64-byte pieces of a k-row, half a line
// each); 16 x 4096 -> 4096 13.0 -> 8.3; 257 x 1536 -> 384 7.6 -> 6.1; 70 x 768 -> 768 5.3 -> 4.2; and with one chain 177 x 80 -> 200
// 4.6 -> 4.05, 80 x 192 -> 128 4.0 -> 3.8, 692 x 320 -> 192 5.1 -> 4.5 (12 % at the median of 80 shapes).
// One workgroup a CU at most: past that the ring's larger tile moves fewer bytes (1370 x 1536 -> 384 8.1 against 11.4 here), and half
// the stages, two workgroups a CU, gained 0.1 % over the shapes of the planner's fit.
//
// LDS layout of a stage: A rows of 256 bytes, then B ([N][K]: the same; [K][N]: 128 rows of 64 bytes).  Sixteen-byte chunks are permuted
// inside their row: K-contiguous row r holds chunk c at c ^ (r % 16), [K][N] row k at c ^ (k % 4).
//
// CONV: B is the patch matrix of a convolution (ConvGather), its rows' offsets fixed and the tap moving.  A 128-deep stage may hold
// eight taps (sixteen channels each), and the permutation gives a lane another chunk in each of four requests in a row.  Two loader
// waves take two of the four each, request by request, so a lane keeps two (tap, channel) states, advanced by whole taps and what is
// left of a stage: some twelve instructions each for the 400 clocks of a stage.  K is split whatever its depth: nothing promises one
// chain of sums of a convolution.
// Against the 64 x 64 ring, both behind conv_pad_kernel, in us (workgroups): 144 x 34 x 60 -> 32, 7 x 7 stride 4 (5) 29.5 -> 20.3;
// 96 x 22 x 23 -> 96, 5 x 5 (48) 15.5 -> 11.6; 256 x 29 x 11 -> 384, 5 x 5 (120) 29.1 -> 23.6; 256 x 30 x 112 -> 64, 3 x 3 (210) 13.9 -> 12.4.
// 43 convolutions of at most 256 workgroups, 2304 deep in the middle: 0.81 of the time, geometric mean, none slower.
constexpr int S = 8;                      // stages of the ring: 128 KB

template <int NW, int CHAINS, bool B_KN, bool CONV = false>
__global__ __launch_bounds__((NW + 3) * 64, 2) void gemm_deep_kernel(GemmArgs p) {
    static_assert(!(CONV && B_KN), "a patch row is K-contiguous");
    constexpr int BM = 32, BN = 32, BK = 128, AHEAD = 5;
    constexpr int STEPS = 8 / NW;                         // a matrix wave's steps of a stage
    constexpr int A_BYTES = BM * BK * 2, STAGE_BYTES = 2 * A_BYTES;
    extern __shared__ __align__(16) char smem[];
    stage_args(p);
    const int tid = threadIdx.x, lane = tid & 63, wave = __builtin_amdgcn_readfirstlane(tid >> 6);
    int tm_, tn_;
    tile_of(p, tm_, tn_);
    const int m0 = __builtin_amdgcn_readfirstlane(tm_ * BM), n0 = __builtin_amdgcn_readfirstlane(tn_ * BN);
    const long bz = blockIdx.y;
    const int nk = (p.K + BK - 1) / BK;
    const uint32_t lds0 = (uint32_t)(uintptr_t)(__attribute__((address_space(3))) char *)smem;
    auto barrier = [&]() {
        asm volatile("" ::: "memory");
        __builtin_amdgcn_s_barrier();
        asm volatile("" ::: "memory");
    };

    if (__builtin_expect(wave >= NW, 1)) {
        nothing_pending();
        auto load_all = [&](auto IS_A_) __attribute__((always_inline)) {
            constexpr bool IS_A = decltype(IS_A_)::value, ROWS = IS_A || !B_KN, PATCH = CONV && !IS_A;
            // 1 KB requests of a stage, a run of RUN in a row sharing an LDS address.  PATCH: 2 half + {0, 1, 4, 5}
            constexpr int LPW = PATCH ? 4 : 8, RUN = PATCH ? 2 : 4;
            const int half = PATCH ? wave - (NW + 1) : 0;
            uint32_t off[LPW];
            int kpos[LPW];                                // first k of the lane's chunk
            const long ld2 = (IS_A ? p.ldA : p.ldB) * 2;
            const int r0 = IS_A ? m0 : n0, rows = IS_A ? p.M : p.N;
#pragma unroll
            for (int i = 0; i < LPW; i++) {
                if constexpr (PATCH) {
                    const int slot = 2 * half + (i & 1) + 4 * (i >> 1), r = 4 * slot + (lane >> 4), c = (lane & 15) ^ (r & 15);
                    unsigned ow;
                    const unsigned oh = divide(min(r0 + r, rows - 1), p.cv.OW, p.cv.div_OW, ow);
                    off[i] = (oh * p.cv.pix_y + ow * p.cv.pix_x) * 2u + (c & 1) * 16;
                    kpos[i] = c * 8;
                } else if constexpr (ROWS) {              // request i: rows 4 i .. 4 i + 3; past the edge the last one again
                    const int r = 4 * i + (lane >> 4), c = (lane & 15) ^ (r & 15);
                    off[i] = (uint32_t)((min(r0 + r, rows - 1) - r0) * ld2) + c * 16;
                    kpos[i] = c * 8;
                } else {                                  // k-rows 16 i .. 16 i + 15; past the edge the last chunk again
                    const int k = 16 * i + (lane >> 2), c = (lane & 3) ^ (k & 3);
                    off[i] = (uint32_t)(k * ld2) + max(0, min(c * 8, p.NB - 8 - n0)) * 2;
                    kpos[i] = k;
                }
            }
            constexpr int LOW = 1024 * (RUN - 1);         // a request's immediate offset moves source and destination alike: gemm_ring_kernel
#pragma unroll
            for (int i = 0; i < LPW; i++) off[i] += LOW - 1024 * (i & (RUN - 1));
            const char *org = (IS_A ? reinterpret_cast<const char *>(p.A + bz * p.sA + (long)m0 * p.ldA)
                                    : PATCH ? reinterpret_cast<const char *>(p.cv.xp + bz * p.cv.img)
                                    : reinterpret_cast<const char *>(p.B + bz * p.sB + (B_KN ? (long)n0 : (long)n0 * p.ldB))) - LOW;
            const long step = PATCH ? 0 : ROWS ? BK * 2 : (long)BK * p.ldB * 2;
            const uint32_t lds1 = lds0 + (IS_A ? 0 : A_BYTES) + half * 2048;
            // PATCH: channel, tap column and byte offset, from the pixel, of the pair of chunks that requests i with i % 2 = t take next
            const int taps = PATCH ? BK / p.cv.C : 0, rest = PATCH ? BK - taps * p.cv.C : 0, rows_max = PATCH ? (taps + p.cv.KW) / p.cv.KW : 0;
            const int tap_step = p.cv.tap_x * 2, over_step = (p.cv.tap_x - p.cv.C) * 2, row_step = (p.cv.tap_y - p.cv.KW * p.cv.tap_x) * 2;
            const int stage_step = taps * tap_step + rest * 2;
            int ch[2], kw[2];
            uint32_t at[2] = {0u, 0u};
            if constexpr (PATCH) {
#pragma unroll
                for (int t = 0; t < 2; t++) {
                    unsigned c, w;
                    const unsigned tap = divide(kpos[t] & ~15, p.cv.C, p.cv.div_C, c), kh = divide(tap, p.cv.KW, p.cv.div_KW, w);
                    ch[t] = c; kw[t] = w;
                    at[t] = (c + kh * p.cv.tap_y + w * p.cv.tap_x) * 2u;
                }
            }
            int next = 0;                                 // the stage of K requested next, and where it goes
            uint32_t stage = 0;
            auto request = [&]() __attribute__((always_inline)) {
                if ((next + 1) * BK <= p.K) {             // uniform
#pragma unroll
                    for (int q = 0; q < LPW; q += RUN)
                        if constexpr (PATCH)
                            asm volatile("s_mov_b32 m0, %0\n\t"
                                         "s_nop 0\n\t"
                                         "global_load_lds_dwordx4 %1, %3\n\t"
                                         "global_load_lds_dwordx4 %2, %3 offset:1024" ::"s"(lds1 + stage + q * 2048),
                                         "v"(off[q] + at[0]), "v"(off[q + 1] + at[1]), "s"(org) : "memory");
                        else asm volatile("s_mov_b32 m0, %0\n\t"
                                     "s_nop 0\n\t"
                                     "global_load_lds_dwordx4 %1, %5\n\t"
                                     "global_load_lds_dwordx4 %2, %5 offset:1024\n\t"
                                     "global_load_lds_dwordx4 %3, %5 offset:2048\n\t"
                                     "global_load_lds_dwordx4 %4, %5 offset:3072" ::"s"(lds1 + stage + q * 1024),
                                     "v"(off[q]), "v"(off[q + 1]), "v"(off[q + 2]), "v"(off[q + 3]), "s"(org) : "memory");
                } else {                                  // the stage that K ends in: chunks past it come from the zeros
#pragma unroll
                    for (int i = 0; i < LPW; i++) {
                        const char *from = next * BK + kpos[i] < p.K ? org + (off[i] + (PATCH ? at[i & 1] : 0u)) + 1024 * (i & (RUN - 1)) : reinterpret_cast<const char *>(deep_zero_words);
                        const uint32_t to = PATCH ? (i & 1) * 1024 + (i >> 1) * 4096 : i * 1024;
                        asm volatile("s_mov_b32 m0, %1\n\ts_nop 0\n\tglobal_load_lds_dwordx4 %0, off" ::"v"(from), "s"(lds1 + stage + to) : "memory");
                    }
                }
                if constexpr (PATCH) {
#pragma unroll
                    for (int t = 0; t < 2; t++) {
                        ch[t] += rest;
                        const bool over = ch[t] >= p.cv.C;
                        ch[t] -= over ? p.cv.C : 0;
                        kw[t] += taps + (over ? 1 : 0);
                        at[t] += stage_step + (over ? over_step : 0);
                        for (int r = 0; r < rows_max; r++) {      // on to the taps of the next rows
                            const bool row = kw[t] >= p.cv.KW;
                            kw[t] -= row ? p.cv.KW : 0;
                            at[t] += row ? row_step : 0;
                        }
                    }
                }
                org += step;
                next++;
                stage = stage == (S - 1) * STAGE_BYTES ? 0u : stage + STAGE_BYTES;
            };
            // all but the newest `newer` stages' requests have landed
            auto landed = [&](int newer) {
                switch (newer) {
                case 0: asm volatile("s_waitcnt vmcnt(0)" ::: "memory"); break;
                case 1: asm volatile("s_waitcnt vmcnt(%0)" ::"n"(LPW) : "memory"); break;
                case 2: asm volatile("s_waitcnt vmcnt(%0)" ::"n"(2 * LPW) : "memory"); break;
                case 3: asm volatile("s_waitcnt vmcnt(%0)" ::"n"(3 * LPW) : "memory"); break;
                default: asm volatile("s_waitcnt vmcnt(%0)" ::"n"(4 * LPW) : "memory"); break;
                }
            };
            static_assert(AHEAD <= 5 && AHEAD < S, "landed() counts to four; a stage being read while the others are on their way");
            const int ahead = min(AHEAD, nk);
            for (int kt = 0; kt < ahead; kt++) request();
            landed(ahead - 1);
            barrier();                                    // stage 0 has landed
            int kt = 0;
            for (; next < nk; kt++) {
                asm volatile("s_waitcnt vmcnt(%0)" ::"n"((AHEAD - 2) * LPW) : "memory");      // stage kt + 1 has landed
                barrier();
                request();
            }
            for (; kt + 1 < nk; kt++) {
                landed(nk - (kt + 2));
                barrier();
            }
        };
        if (!CONV && wave == NW + 2) lnf_stats_wave<BM, BN, false, 4>(p, reinterpret_cast<float2v *>(smem + S * STAGE_BYTES), m0, n0, bz, lane, nk, barrier);
        else if (wave == NW) load_all(std::true_type{});
        else load_all(std::false_type{});
        return;
    }

    // fragment addresses of this wave's steps of a stage, `wave` and every NW-th after it
    const int frow = lane & 31, h = lane >> 5, k3 = (lane & 15) >> 2, n = ((lane >> 4) & 1) * 16 + (lane & 3) * 4;
    uint32_t aoff[STEPS], boff[STEPS];
#pragma unroll
    for (int s = 0; s < STEPS; s++) {
        const int ks = wave + NW * s;
        aoff[s] = frow * 256 + (((2 * ks + h) ^ (frow & 15)) * 16);
        if constexpr (!B_KN) boff[s] = A_BYTES + aoff[s];
        else boff[s] = A_BYTES + (ks * 16 + h * 8 + k3) * BN * 2 + (((n >> 3) ^ k3) * 16) + (n & 7) * 2;
    }
    half8v fa[2][STEPS], fb[2][STEPS];
    auto fetch = [&](auto SET, int kt) __attribute__((always_inline)) {
        constexpr int set = decltype(SET)::value;
        const char *st = smem + (kt % S) * STAGE_BYTES;
#pragma unroll
        for (int s = 0; s < STEPS; s++) {
            fa[set][s] = *reinterpret_cast<const half8v *>(st + aoff[s]);
            if constexpr (!B_KN) fb[set][s] = *reinterpret_cast<const half8v *>(st + boff[s]);
            else {
                const char *b = st + boff[s];
                const short4v lo = __builtin_amdgcn_ds_read_tr16_b64_v4i16((__attribute__((address_space(3))) short4v *)b);
                const short4v hi = __builtin_amdgcn_ds_read_tr16_b64_v4i16((__attribute__((address_space(3))) short4v *)(b + 4 * BN * 2));
                const short8v both = {lo[0], lo[1], lo[2], lo[3], hi[0], hi[1], hi[2], hi[3]};
                fb[set][s] = __builtin_bit_cast(half8v, both);
            }
        }
    };
    float16v acc[CHAINS];
#pragma unroll
    for (int s = 0; s < CHAINS; s++)
#pragma unroll
        for (int r = 0; r < 16; r++) acc[s][r] = 0.0f;
    auto products = [&](auto SET) {
        constexpr int set = decltype(SET)::value;
#pragma unroll
        for (int s = 0; s < STEPS; s++) {
            constexpr int first = set * STEPS;            // (four chains: odd and even stages' steps apart)
            acc[(first + s) % CHAINS] = __builtin_amdgcn_mfma_f32_32x32x16_f16(fb[set][s], fa[set][s], acc[(first + s) % CHAINS], 0, 0, 0);
        }
    };

    // what the store needs of memory, while the first stages are on their way
    half4v cb[1][4];
    ResidualAhead<32> res;
    if (wave == 0) {
        load_col_bias<1, 32>(p, cb, n0, 0, lane, bz);
        res.request(p, m0, n0, lane, bz);
    }
    barrier();
    using I0 = std::integral_constant<int, 0>;
    using I1 = std::integral_constant<int, 1>;
    // past the barrier stage kt + 1 has landed and stage kt - 1 is free for the loaders
    auto turn = [&](auto SET, auto NEXT, int kt) __attribute__((always_inline)) {
        barrier();
        fetch(NEXT, kt + 1);
        __builtin_amdgcn_sched_barrier(0);                // the reads go out ahead of the products,
        products(SET);
        __builtin_amdgcn_sched_barrier(0);                // which stay ahead of the next barrier: by then this stage has been read
    };
    if (nk & 1) {                                         // an odd stage comes first: gemm_ring_kernel
        fetch(I1{}, 0);
        if (nk > 1) turn(I1{}, I0{}, 0);
    } else fetch(I0{}, 0);
    int kt = nk & 1;
    for (; kt + 2 < nk; kt += 2) {
        turn(I0{}, I1{}, kt);
        turn(I1{}, I0{}, kt + 1);
    }
    if (nk > 1) turn(I0{}, I1{}, kt);
    products(I1{});

    // Partial tiles, then the store's staging, in memory that the last two stages (which slower waves may still read) do not take
    constexpr int PARTS = (NW - 1) * 4096, ROOM = PARTS + 2 * 32 * 40 * 2;
    char *room = smem;
    static_assert((S - 1) * STAGE_BYTES - ROOM >= ROOM + STAGE_BYTES, "above the last stage, or below the one before it");
    const int l = (nk - 1) % S;
    if ((l + 1) * STAGE_BYTES + ROOM <= S * STAGE_BYTES) room = smem + (l + 1) * STAGE_BYTES;
    float16v own[1][1];
#pragma unroll
    for (int r = 0; r < 16; r++) own[0][0][r] = CHAINS == 4 ? (acc[0][r] + acc[1 % CHAINS][r]) + (acc[2 % CHAINS][r] + acc[3 % CHAINS][r]) : CHAINS == 2 ? acc[0][r] + acc[1 % CHAINS][r] : acc[0][r];
    if constexpr (NW > 1) {
        float *part = reinterpret_cast<float *>(room);
        if (wave > 0) {
#pragma unroll
            for (int r4 = 0; r4 < 4; r4++) {
                const float4v q = {own[0][0][4 * r4], own[0][0][4 * r4 + 1], own[0][0][4 * r4 + 2], own[0][0][4 * r4 + 3]};
                *reinterpret_cast<float4v *>(part + (wave - 1) * 1024 + r4 * 256 + lane * 4) = q;
            }
        }
        asm volatile("s_waitcnt lgkmcnt(0)" ::: "memory");
        barrier();
        if (wave > 0) return;
        float4v got[NW - 1][4];
#pragma unroll
        for (int w = 0; w < NW - 1; w++)
#pragma unroll
            for (int r4 = 0; r4 < 4; r4++) got[w][r4] = *reinterpret_cast<const float4v *>(part + w * 1024 + r4 * 256 + lane * 4);
#pragma unroll
        for (int r = 0; r < 16; r++) own[0][0][r] = (own[0][0][r] + got[0][r >> 2][r & 3]) + (got[1][r >> 2][r & 3] + got[2][r >> 2][r & 3]);
    }
    LnFold<1> ln;
    if (p.lnf_stats) {
        const float2v *slot = reinterpret_cast<const float2v *>(smem + S * STAGE_BYTES);
        const float2v v = slot[frow];
        ln.on = true; ln.col = reinterpret_cast<const float *>(slot + BM); ln.bn = BN; ln.r[0] = v[0]; ln.rmu[0] = v[1];
    }
    store_tile<1, 1, 32, 32, 1, S * STAGE_BYTES>(p, own, cb, room + PARTS, m0, n0, 0, 0, 0, lane, bz, ln, &res);
}

constexpr int DEEP_LDS_BYTES = S * 2 * 32 * 128 * 2 + 2 * 32 * 8;       // the stages; rows' and columns' parts of a folded norm

template <int CHAINS>
int launch_deep_patches(const GemmArgs &a, int64_t nbatch, hipStream_t st) {
    hipLaunchKernelGGL((gemm_deep_kernel<4, CHAINS, false, true>), dim3((unsigned)(a.tiles_m * a.tiles_n), (unsigned)nbatch), dim3(7 * 64), DEEP_LDS_BYTES, st, a);
    return hipGetLastError() == hipSuccess ? MI_OK : MI_ERROR_LAUNCH;
}
template <int NW, int CHAINS>
int launch_deep(const GemmArgs &a, bool b_kn, int64_t nbatch, hipStream_t st) {
    const dim3 grid((unsigned)(a.tiles_m * a.tiles_n), (unsigned)nbatch), block((NW + (a.lnf_stats ? 3 : 2)) * 64);
    if (b_kn) hipLaunchKernelGGL((gemm_deep_kernel<NW, CHAINS, true>), grid, block, DEEP_LDS_BYTES, st, a);
    else      hipLaunchKernelGGL((gemm_deep_kernel<NW, CHAINS, false>), grid, block, DEEP_LDS_BYTES, st, a);
    return hipGetLastError() == hipSuccess ? MI_OK : MI_ERROR_LAUNCH;
}
template <int NW, int CHAINS>
int raise_deep() { return raise_lds(gemm_deep_kernel<NW, CHAINS, true>, DEEP_LDS_BYTES) | raise_lds(gemm_deep_kernel<NW, CHAINS, false>, DEEP_LDS_BYTES); }

}  // namespace

// per-lane load offsets are 32-bit byte offsets from the tile's origin
bool mi_deep_takes(int64_t ldA, int64_t ldB) { return 32 * ldA * 2 < (1ll << 31) && 128 * ldB * 2 < (1ll << 31); }

int mi_deep_launch(const GemmArgs &args, bool split_k, bool b_kn, int64_t nbatch, hipStream_t st) {
    GemmArgs a = args;
    set_tiles(a, 32, 32);
    a.vec_store = rows_vec16(a);
    if (a.cv.xp) {
        if (b_kn || a.cv.img > MI_PATCH_IMAGE_MAX || (int64_t)32 * a.ldA * 2 >= (1ll << 31)) return MI_DECLINE_EXTENT;
        return a.K > 4096 ? launch_deep_patches<4>(a, nbatch, st) : launch_deep_patches<2>(a, nbatch, st);
    }
    if (!mi_deep_takes(a.ldA, a.ldB)) return MI_DECLINE_EXTENT;
    // Past K = 4096 such calls had twelve to twenty chains, as slices of K on the ring; short of it eight are as good as what they had, and
    // the second pair of accumulators costs 0.05 to 0.1 us (50 x 3224 -> 992 6.67 | 6.75).
    // Up to eight rows replace K-slices of [K][F] weights, whose error eight chains exceed from K = 1280 on (9.4e-8 | 9.7e-8, sixteen 8.3e-8).
    if (!split_k) return launch_deep<1, 1>(a, b_kn, nbatch, st);
    return a.K > 4096 || (a.M <= 8 && a.K > 768) ? launch_deep<4, 4>(a, b_kn, nbatch, st) : launch_deep<4, 2>(a, b_kn, nbatch, st);
}

int mi_deep_init() {
    return raise_lds(gemm_deep_kernel<4, 2, false, true>, DEEP_LDS_BYTES) | raise_lds(gemm_deep_kernel<4, 4, false, true>, DEEP_LDS_BYTES) |
           raise_deep<4, 4>() | raise_deep<4, 2>() | raise_deep<1, 1>();
}
