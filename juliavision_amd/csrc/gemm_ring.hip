// fp16 GEMM for gfx950, 64 x 64 tiles over a ring of direct-to-LDS stages: grids too small for the four-wave kernel.
#include "gemm_common.hpp"

// Sixteen zero bytes for loads of chunks past the end of K.
static __device__ __align__(16) unsigned ring_zero_words[4];

namespace {

// A workgroup owns a 64 x 64 tile, each of its four matrix waves a 32 x 32 block of it; two loader waves keep the ring filled, a
// seventh takes in a folded norm's statistics.
//
// What bounds such a tile is the CU's LDS and vector-memory path, not the matrix cores: per 64-deep tile 256 clocks of 64 B/clock
// loads and 384 of LDS (16 KB in, 32 KB of fragments out) for 128 clocks of MFMAs.  Measured, a tile takes 320 to 400 clocks; the
// register-staged kernel's same tile was at 480 to 670, because its loads pass through registers and its waits are the
// compiler's.  In launches of one tile a CU the ends cost as much as the loop, and that is where the arrangement comes from
// (clocks at 1370 x 1536 -> 384, 132 workgroups; before, with waves that split K's steps and a ring filled before the first
// product): first request 2040 -> 840 (stage_args, tile_of), products begin 4620 -> 2600 (AHEAD tiles asked for, not the whole
// ring), sum of the waves' partial tiles 2020 -> none, store 2030 -> 1270 (its residual comes with the first tiles).  8.3 -> 7.3 us
// a launch; 1370 x 384 -> 384, where four waves that split K lost to the register-staged kernel, 4.8 -> 4.6, 76 x 1024 -> 3072
// 6.7 -> 5.9, 2056 x 1536 -> 384 8.7 -> 7.8.  Waves that split K read
// 16 KB of fragments a tile instead of 32 and gain from some 45 tiles of K on in the smallest grids (32 x 3456 -> 448 10.3 against
// 11.2 us); over 150 shapes they are 6 % behind.
//
// LDS layout of a stage: A rows of 128 bytes, then B ([N][K]: rows of 128 bytes; [K][N]: 64 rows of BN halves).  Direct loads
// cannot pad, so 16-byte chunks are permuted inside their row: K-contiguous row r holds chunk c at c ^ (r % 8 ^ r / 8 % 2),
// [K][N] row k holds chunk c at c ^ (k % 4 * BN / 32) -- the four rows of a transposing read in four bank groups.
// Chunks past K are read from a page of zeros, so K needs only to be a multiple of 8.
//
// CONV: B is the patch matrix of a convolution (ConvGather).  Its rows' offsets are as fixed as an ordinary operand's; what moves
// from tile to tile is the tap, for all lanes alike where C is a multiple of 64, by the lane's pair of chunks otherwise.
//
// Chains of fp32 sums an element, the 16-deep step ks of every tile in chain ks % chains: four from K = 513 on and for patches.  One
// chain has 1.8 times the error of four (fp32 results against 64 bits: K = 768 1.78e-7 | 1.00e-7, 1536 2.49e-7 | 1.33e-7, 5120 4.55e-7 |
// 2.32e-7) at the same time (1000 x 1536 -> 1000 8.13 | 8.17 us, 1000 x 5120 -> 1000 22.3 | 20.8).  One up to there, in the order of
// every other tile: a call that folds a layer norm promises the bits of the norm and this GEMM apart.  One too for ordinary operands
// past one workgroup a CU, whose registers are short.  Both loops are in one kernel: as two, a model that alternates between them paid
// for each one's cold instructions (ViT-S of 1370 tokens, 24 such launches: 529 us as two, 521 so, 514 with one chain throughout).
template <int S, bool B_KN, bool CONV = false>
__global__ __launch_bounds__(4 * 64 + (CONV ? 128 : 192), S > 4 ? 2 : CONV ? 3 : 4) void gemm_ring_kernel(GemmArgs p) {
    constexpr int BM = 64, BN = 64, BK = 64, NW = 4;
    constexpr int SLOTS_A = BM / 8, SLOTS = (BM + BN) / 8;        // 1 KB requests of a stage
    constexpr int STAGE_BYTES = SLOTS * 1024, A_BYTES = SLOTS_A * 1024;
    static_assert(!(CONV && B_KN), "a patch row is K-contiguous");
    static_assert(S >= 3, "a stage being read, one landed, one on its way");
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

    if (__builtin_expect(wave >= NW, 1)) {                // (laid out first: what the launch waits for)
        // The loaders, one for each operand.  A matrix wave that issued its share of the requests stood at those instructions
        // with its products behind them (800 clocks a 64 x 64 tile), and a loader is quick only if a request costs it next
        // to nothing: a wave issues an instruction every four to eight clocks, so the lane's byte offset from the tile's
        // origin is fixed, the origin and the LDS address move in scalar registers, and the steady state has no branch.
        // ROLE: 0 A, 1 B, 2 B a patch matrix whose tiles lie in one tap each, 3 any other patch matrix
        auto load_all = [&](auto ROLE) {
            constexpr bool IS_A = decltype(ROLE)::value == 0, PATCH = decltype(ROLE)::value >= 2, ONE_TAP = decltype(ROLE)::value == 2;
            constexpr int LPW = IS_A ? SLOTS_A : SLOTS - SLOTS_A;      // 1 KB requests of a tile
            static_assert((S - 2) * LPW <= 63, "vmcnt is a 6-bit counter");
            uint32_t off[LPW];
            int kpos[LPW];                                // first k of the lane's chunk
            // Request i covers rows 8 i .. 8 i + 7 (K-contiguous) or 512 / BN k-rows; the permutation has period two in i, so
            // inside the operand an offset is one of two plus i times a constant.
            constexpr bool ROWS = IS_A || !B_KN;
            const int pos = lane & 7, sub = lane >> 3;
            const long ld2 = (IS_A ? p.ldA : p.ldB) * 2;
            if (ROWS) {
                const int r0 = IS_A ? m0 : n0, rows = IS_A ? p.M : p.N, c = pos ^ sub;
                const uint32_t even = (uint32_t)(sub * ld2) + c * 16, odd = even + ((c ^ 1) - c) * 16, step8 = (uint32_t)(8 * ld2);
                const bool inside = r0 + (IS_A ? BM : BN) <= rows;                    // uniform
                if constexpr (PATCH) {
                    // rows are pixels, eight apart from request to request: one division, then steps
                    const int last = rows - 1, last_y = last / p.cv.OW, last_off = last_y * p.cv.pix_y + (last - last_y * p.cv.OW) * p.cv.pix_x;
                    int n = r0 + sub, oh = n / p.cv.OW, ow = n - oh * p.cv.OW;
#pragma unroll
                    for (int i = 0; i < LPW; i++) {
                        const int ci = c ^ (i & 1);
                        off[i] = (uint32_t)(n < rows ? oh * p.cv.pix_y + ow * p.cv.pix_x : last_off) * 2u + (ONE_TAP ? ci : ci & 1) * 16;
                        kpos[i] = ci * 8;
                        n += 8; ow += 8;
                        while (ow >= p.cv.OW) { ow -= p.cv.OW; oh++; }
                    }
                } else
#pragma unroll
                for (int i = 0; i < LPW; i++) {
                    off[i] = ((i & 1) ? odd : even) + i * step8;
                    if (!inside) off[i] = (uint32_t)((min(r0 + 8 * i + sub, rows - 1) - r0) * ld2) + (c ^ (i & 1)) * 16;
                    kpos[i] = (c ^ (i & 1)) * 8;
                }
            } else {
                constexpr int CPR = BN / 8, PER = 64 / CPR;                           // chunks of a k-row, k-rows of a request
                const int k = lane / CPR, c = (lane % CPR) ^ ((k & 3) * (BN / 32));
                // columns past the edge re-read the last chunk
                const uint32_t first = (uint32_t)(k * ld2) + max(0, min(c * 8, p.NB - 8 - n0)) * 2, stepk = (uint32_t)(PER * ld2);
                static_assert(PER % 4 == 0, "a request's k-rows start on a multiple of four");
#pragma unroll
                for (int i = 0; i < LPW; i++) {
                    off[i] = first + i * stepk;
                    kpos[i] = k + i * PER;
                }
            }
            const char *org = IS_A ? reinterpret_cast<const char *>(p.A + bz * p.sA + (long)m0 * p.ldA)
                              : PATCH ? reinterpret_cast<const char *>(p.cv.xp + bz * p.cv.img)
                                      : reinterpret_cast<const char *>(p.B + bz * p.sB + (B_KN ? (long)n0 : (long)n0 * p.ldB));
            // PATCH: where the next tile's first channel lies (ONE_TAP: the same for every lane, kept in `org`), or this lane's
            // pair of chunks of it (C % 16 == 0: a pair never straddles two taps)
            const int tap_step = (p.cv.tap_x - p.cv.C) * 2, row_step = (p.cv.tap_y - p.cv.KW * p.cv.tap_x) * 2;
            int ch = 0, kw = 0, at = 0;
            const int wraps = PATCH && !ONE_TAP ? (BK + p.cv.C - 1) / p.cv.C : 1;
            auto advance = [&](int by) {
                ch += by;
                at += by * 2;
                for (int w = 0; w < wraps; w++) {         // past the tap's channels: on to the next tap
                    const bool over = ch >= p.cv.C;
                    kw += over ? 1 : 0;
                    const bool row = kw == p.cv.KW;
                    at += (over ? tap_step : 0) + (row ? row_step : 0);
                    ch -= over ? p.cv.C : 0;
                    kw = row ? 0 : kw;
                }
            };
            if (PATCH && !ONE_TAP) advance(((pos ^ sub) & 6) * 8);
            const long step = IS_A || !B_KN ? BK * 2 : (long)BK * p.ldB * 2;
            const uint32_t lds1 = lds0 + (IS_A ? 0 : A_BYTES);
            int next = 0;                                 // the tile requested next, and its stage
            uint32_t stage = 0;
            // A request's immediate offset moves its source and its destination alike: four requests share an LDS address, with the
            // lane's offset lowered by what the immediate adds and the origin by the most of it, so that no offset is negative.
            constexpr int LOW = 3072;
#pragma unroll
            for (int i = 0; i < LPW; i++) off[i] += LOW - 1024 * (i & 3);
            org -= LOW;
            auto request = [&]() {
                const uint32_t add = PATCH && !ONE_TAP ? (uint32_t)at : 0u;
                const char *from_org = ONE_TAP ? org + at : org;
                if ((next + 1) * BK <= p.K) {             // uniform
#pragma unroll
                    for (int q = 0; q < LPW; q += 4)
                        asm volatile("s_mov_b32 m0, %0\n\t"
                                     "s_nop 0\n\t"
                                     "global_load_lds_dwordx4 %1, %5\n\t"
                                     "global_load_lds_dwordx4 %2, %5 offset:1024\n\t"
                                     "global_load_lds_dwordx4 %3, %5 offset:2048\n\t"
                                     "global_load_lds_dwordx4 %4, %5 offset:3072" ::"s"(lds1 + stage + q * 1024),
                                     "v"(off[q] + add), "v"(off[q + 1] + add), "v"(off[q + 2] + add), "v"(off[q + 3] + add), "s"(from_org) : "memory");
                } else {                                  // the tile that K ends in: chunks past it come from the zeros
#pragma unroll
                    for (int i = 0; i < LPW; i++) {
                        const char *from = next * BK + kpos[i] < p.K ? from_org + (off[i] + add) + 1024 * (i & 3) : reinterpret_cast<const char *>(ring_zero_words);
                        asm volatile("s_mov_b32 m0, %1\n\ts_nop 0\n\tglobal_load_lds_dwordx4 %0, off" ::"v"(from), "s"(lds1 + stage + i * 1024) : "memory");
                    }
                }
                if constexpr (PATCH) advance(BK);
                else org += step;
                next++;
                stage = stage == (S - 1) * STAGE_BYTES ? 0u : stage + STAGE_BYTES;
            };
            // all but the newest `newer` tiles' requests have landed
            auto landed = [&](int newer) {
                switch (newer) {
                case 0: asm volatile("s_waitcnt vmcnt(0)" ::: "memory"); break;
                case 1: asm volatile("s_waitcnt vmcnt(%0)" ::"n"(LPW) : "memory"); break;
                case 2: asm volatile("s_waitcnt vmcnt(%0)" ::"n"(S > 3 ? 2 * LPW : 0) : "memory"); break;
                case 3: asm volatile("s_waitcnt vmcnt(%0)" ::"n"(S > 4 ? 3 * LPW : 0) : "memory"); break;
                case 4: asm volatile("s_waitcnt vmcnt(%0)" ::"n"(S > 5 ? 4 * LPW : 0) : "memory"); break;
                case 5: asm volatile("s_waitcnt vmcnt(%0)" ::"n"(S > 6 ? 5 * LPW : 0) : "memory"); break;
                default: asm volatile("s_waitcnt vmcnt(%0)" ::"n"(S > 7 ? 6 * LPW : 0) : "memory"); break;
                }
            };
            static_assert(S <= 8, "landed() counts to six");
            // Products start when the first AHEAD tiles have been asked for, at 256 clocks a tile: enough of them to cover a trip to
            // memory, and no more.
            constexpr int AHEAD = S > 4 ? 5 : S - 1;
            const int ahead = min(AHEAD, nk);
            for (int kt = 0; kt < ahead; kt++) request();
            landed(ahead - 1);
            barrier();                                    // tile 0 has landed
            int kt = 0;
            for (; next < nk; kt++) {
                asm volatile("s_waitcnt vmcnt(%0)" ::"n"((AHEAD - 2) * LPW) : "memory");      // tile kt + 1 has landed
                barrier();
                request();
            }
            for (; kt + 1 < nk; kt++) {
                landed(nk - (kt + 2));
                barrier();
            }
        };
        if (wave == NW + 2) lnf_stats_wave<BM, BN, false>(p, reinterpret_cast<float2v *>(smem + S * STAGE_BYTES), m0, n0, bz, lane, nk, barrier);
        else if (wave == NW) load_all(std::integral_constant<int, 0>{});
        else if constexpr (!CONV) load_all(std::integral_constant<int, 1>{});
        else if (p.cv.C % 64 == 0) load_all(std::integral_constant<int, 2>{});
        else load_all(std::integral_constant<int, 3>{});
        return;
    }

    // fragment addresses of this wave's 32 x 32 block, a 16-deep step of a tile each
    constexpr int NKS = BK / 16;
    const int sm = wave & 1, sn = wave >> 1;
    const int frow = lane & 31, h = lane >> 5, aswz = (frow & 7) ^ ((frow >> 3) & 1), k3 = (lane & 15) >> 2;
    const int n = sn * 32 + ((lane >> 4) & 1) * 16 + (lane & 3) * 4;
    const uint32_t noff = (uint32_t)((((n >> 3) ^ (k3 * (BN / 32))) * 16) + (n & 7) * 2);
    uint32_t aoff[NKS], boff[NKS];
#pragma unroll
    for (int ks = 0; ks < NKS; ks++) {
        const uint32_t chunk = (uint32_t)(((2 * ks + h) ^ aswz) * 16);
        aoff[ks] = (sm * 32 + frow) * 128 + chunk;
        if constexpr (!B_KN) boff[ks] = A_BYTES + (sn * 32 + frow) * 128 + chunk;
        else boff[ks] = (uint32_t)(A_BYTES + (ks * 16 + h * 8 + k3) * BN * 2) + noff;
    }
    half8v fa[2][NKS], fb[2][NKS];
    auto fetch = [&](auto SET, int kt) {
        constexpr int set = decltype(SET)::value;
        const char *st = smem + (kt % S) * STAGE_BYTES;
#pragma unroll
        for (int ks = 0; ks < NKS; ks++) {
            fa[set][ks] = *reinterpret_cast<const half8v *>(st + aoff[ks]);
            if constexpr (!B_KN) fb[set][ks] = *reinterpret_cast<const half8v *>(st + boff[ks]);
            else {
                const char *b = st + boff[ks];
                const short4v lo = __builtin_amdgcn_ds_read_tr16_b64_v4i16((__attribute__((address_space(3))) short4v *)b);
                const short4v hi = __builtin_amdgcn_ds_read_tr16_b64_v4i16((__attribute__((address_space(3))) short4v *)(b + 4 * BN * 2));
                const short8v both = {lo[0], lo[1], lo[2], lo[3], hi[0], hi[1], hi[2], hi[3]};
                fb[set][ks] = __builtin_bit_cast(half8v, both);
            }
        }
    };
    float16v acc[1][1];
    auto products = [&](auto &chain, auto SET) __attribute__((always_inline)) {
        constexpr int ch = sizeof(chain) / sizeof(float16v), set = decltype(SET)::value;
#pragma unroll
        for (int ks = 0; ks < NKS; ks++) chain[ks % ch] = __builtin_amdgcn_mfma_f32_32x32x16_f16(fb[set][ks], fa[set][ks], chain[ks % ch], 0, 0, 0);
    };

    // what the store needs of memory, while the first tiles are on their way
    half4v cb[1][4];
    load_col_bias<1, 32>(p, cb, n0, sn, lane, bz);
    // (two workgroups a CU have no registers to spare for the residual, and each other to hide behind)
    ResidualAhead<32> res;
    if constexpr (S > 4) res.request(p, m0 + sm * 32, n0 + sn * 32, lane, bz);
    const float2v *ln_slot = reinterpret_cast<const float2v *>(smem + S * STAGE_BYTES);
    barrier();
    using I0 = std::integral_constant<int, 0>;
    using I1 = std::integral_constant<int, 1>;
    // Tile kt's fragments are in registers (or on their way) when its turn comes: past the barrier its successor has landed and
    // its predecessor's stage is free for the loaders; the successor's fragments are requested, then its products issued.
    // (The steady state has no branch: where a tile may or may not have a successor, the compiler's wait for its fragments is also
    // one for the successor's, and a turn is longer by an LDS latency.)
    auto turn = [&](auto &chain, auto SET, auto NEXT, int kt) __attribute__((always_inline)) {
        barrier();
        fetch(NEXT, kt + 1);
        __builtin_amdgcn_sched_barrier(0);                // the reads go out ahead of the products,
        products(chain, SET);
        __builtin_amdgcn_sched_barrier(0);                // which stay ahead of the next barrier: by then this tile has been read
    };
    auto tiles = [&](auto CH) __attribute__((always_inline)) {
        constexpr int ch = decltype(CH)::value;
        float16v chain[ch];
#pragma unroll
        for (int s = 0; s < ch; s++)
#pragma unroll
            for (int r = 0; r < 16; r++) chain[s][r] = 0.0f;
        // (an odd tile comes first: one way into the loop and one out of it, or the accumulators are copied between registers)
        if (nk & 1) {
            fetch(I1{}, 0);
            if (nk > 1) turn(chain, I1{}, I0{}, 0);
        } else fetch(I0{}, 0);
        int kt = nk & 1;
        for (; kt + 2 < nk; kt += 2) {
            turn(chain, I0{}, I1{}, kt);
            turn(chain, I1{}, I0{}, kt + 1);
        }
        if (nk > 1) turn(chain, I0{}, I1{}, kt);
        products(chain, I1{});
        acc[0][0] = chain[0];
#pragma unroll
        for (int s = 1; s < ch; s++)
#pragma unroll
            for (int r = 0; r < 16; r++) acc[0][0][r] += chain[s][r];
    };
    if constexpr (CONV) tiles(std::integral_constant<int, 4>{});
    else if (S > 4 && p.K > MI_LNA_KMAX) tiles(std::integral_constant<int, 4>{});
    else tiles(I1{});

    // Past its last barrier of the loop a wave knows that every wave has read all tiles but the last two.  The store's staging keeps
    // clear of their stages where the ring has room for it elsewhere.
    constexpr int STAGING = NW * 2 * 32 * 40 * 2;
    char *staging = smem;
    if constexpr (S > 4) {
        static_assert((S - 1) * STAGE_BYTES - STAGING >= STAGING + STAGE_BYTES, "above the last tile's stage, or below the one before it");
        const int l = (nk - 1) % S;
        if ((l + 1) * STAGE_BYTES + STAGING <= S * STAGE_BYTES) staging = smem + (l + 1) * STAGE_BYTES;
    } else {
        asm volatile("s_waitcnt lgkmcnt(0)" ::: "memory");
        barrier();                                        // every wave has read its last fragments
    }
    LnFold<1> ln;
    if (p.lnf_stats) {
        const float2v v = ln_slot[sm * 32 + frow];
        ln.on = true; ln.col = reinterpret_cast<const float *>(ln_slot + BM); ln.bn = BN; ln.r[0] = v[0]; ln.rmu[0] = v[1];
    }
    store_tile<1, 1, 32, 32, NW, S * STAGE_BYTES>(p, acc, cb, staging, m0, n0, sm, sn, wave, lane, bz, ln, S > 4 ? &res : nullptr);
}

constexpr int ring_lds_bytes(int S) { return S * 2 * 8192 + 2 * 64 * 8; }

template <int S, bool B_KN, bool CONV>
int launch_ring(const GemmArgs &a, int64_t nbatch, hipStream_t st) {
    hipLaunchKernelGGL((gemm_ring_kernel<S, B_KN, CONV>), dim3((unsigned)(a.tiles_m * a.tiles_n), (unsigned)nbatch), dim3(a.lnf_stats ? 448 : 384), ring_lds_bytes(S), st, a);
    return hipGetLastError() == hipSuccess ? MI_OK : MI_ERROR_LAUNCH;
}
template <bool CONV>
int launch_stages(const GemmArgs &a, bool b_kn, bool deep, int64_t nbatch, hipStream_t st) {
    if constexpr (!CONV) {
        if (b_kn) return deep ? launch_ring<8, true, false>(a, nbatch, st) : launch_ring<4, true, false>(a, nbatch, st);
    }
    return deep ? launch_ring<8, false, CONV>(a, nbatch, st) : launch_ring<4, false, CONV>(a, nbatch, st);
}
template <bool B_KN, bool CONV>
int raise_ring() { return raise_lds(gemm_ring_kernel<8, B_KN, CONV>, ring_lds_bytes(8)) | raise_lds(gemm_ring_kernel<4, B_KN, CONV>, ring_lds_bytes(4)); }

}  // namespace

int mi_ring_launch(const GemmArgs &args, bool b_kn, int64_t nbatch, hipStream_t st) {
    GemmArgs a = args;
    set_tiles(a, 64, 64);
    a.vec_store = rows_vec16(a);
    // per-lane load offsets are 32-bit byte offsets from the tile's origin (patches: from the image's)
    if ((int64_t)64 * a.ldA * 2 >= (1ll << 31)) return MI_DECLINE_EXTENT;
    // past one workgroup a CU, half the stages: two of them on a CU (96 -> 384 channels, 3 x 3 stride 2, 27 x 445: 21.1 -> 19.1 us)
    const bool deep = (int64_t)a.tiles_m * a.tiles_n * nbatch <= mi_num_cus();
    if (a.cv.xp) {
        if (b_kn || a.cv.img > MI_PATCH_IMAGE_MAX) return MI_DECLINE_EXTENT;
        return launch_stages<true>(a, false, deep, nbatch, st);
    }
    if ((int64_t)64 * a.ldB * 2 >= (1ll << 31)) return MI_DECLINE_EXTENT;
    return launch_stages<false>(a, b_kn, deep, nbatch, st);
}

int mi_ring_init() {
    return raise_ring<false, true>() | raise_ring<true, false>() | raise_ring<false, false>();
}
