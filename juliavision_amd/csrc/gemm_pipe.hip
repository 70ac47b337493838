// fp16 GEMM for gfx950, the register-staged pipelined kernel: small and medium grids, gathered operands (implicit-GEMM
// convolution), the layer-norm prologue.
#include "gemm_common.hpp"

namespace {

// ------------------------------------------------------------------------------------------
// The software-pipelined kernel for K > 64 (every linear of the encoder configurations).  BM x BN output tile per
// workgroup, WAVES_M x WAVES_N waves, each owning a (BM/WAVES_M) x (BN/WAVES_N) sub-tile as 32x32 MFMA tiles.  The MFMA is
// issued "transposed" (rows = n, columns = m) so that a lane's four consecutive accumulator registers are four
// consecutive n of one output row: an 8-byte fp16 store.  The K loop is written out as a four-phase pipeline per
// 64-deep tile:
//   phase 0: read fragments of k-step 1 | MFMAs of k-step 0   (+ issue the global loads of tile kt+2)
//   phase 1: read fragments of k-step 2 | MFMAs of k-step 1 | write the A part of tile kt+1 to the other LDS buffer
//   phase 2: read fragments of k-step 3 | MFMAs of k-step 2 | write the B part of tile kt+1
//   barrier
//   phase 3: read fragments of k-step 0 of tile kt+1 | MFMAs of k-step 3
// Global loads run two tiles ahead through two register sets, so a load has a
// whole tile of MFMAs to land before its LDS write; the only barrier of a tile sits
// where its successor's first fragment read can be hidden behind the last k-step.
// Two waves per SIMD (8 waves on a 128 x 256 tile) cover each other's waits.
// BMODE: 0 = B is [N][K], 1 = B is [K][N].
// AMODE 1: A is gathered from a channels-last image (NhwcGather); B is then an ordinary [N][K] or [K][N] operand.
// AMODE 2: the rows of A are layer-normalised over K on their way in (K <= 512): before the K loop every wave
// normalises rows of the tile's A panel -- one wave per row, a lane holding eight consecutive k, statistics,
// arithmetic and rounding exactly those of layernorm_vec_kernel -- into an LDS panel [BM][K + 8] that stays resident;
// the K loop then streams B alone and reads its A fragments from the panel.
// KTAIL: K is a multiple of 8 but not of 64.  The last tile's chunks past K re-read the row's last valid chunk (nothing past
// the row is touched) and are zeroed, in both operands, on their way into LDS: two instructions a chunk and load, which is why
// whole tiles keep their own instance.  1544 x 1288 -> 1288 with a residual: 25.7 us through the unpipelined kernel before.
// LNF: the launch has a layer norm folded away (lnf_stats, LnfRows).
template <int BM, int BN, int WAVES_M, int WAVES_N, int BMODE, int AMODE = 0, bool KTAIL = false, bool LNF = false>
__global__ __launch_bounds__(WAVES_M *WAVES_N * 64, LNF && BM * BN == 64 * 128 ? 4 : 2) void gemm_pipe_kernel(GemmArgs p) {
    constexpr bool B_KN = BMODE != 0, LNA = AMODE == 2;
    static_assert(!KTAIL || AMODE == 0, "gathered operands come in whole tiles");
    constexpr int BK = 64, LD = BK + 8, NT = WAVES_M * WAVES_N * 64;
    constexpr int WTM = BM / WAVES_M, WTN = BN / WAVES_N, TM = WTM / 32, TN = WTN / 32;
    constexpr int PA = BM * 8 / NT, PB = BN * 8 / NT;     // 16-byte chunks per thread per tile
    // The [K][N] operand keeps its layout in LDS: BK rows of BN halves, padded by
    // 32 halves so that the four rows a transposing read touches fall in distinct
    // bank groups.  Its MFMA fragments come from ds_read_b64_tr_b16 (see fread).
    constexpr int BLD = BN + 32, CPRB = BN / 8;
    static_assert(PA >= 1 && PB >= 1, "tile too small for this workgroup");
    constexpr int BSZ = B_KN ? BK * BLD : BN * LD;      // halves per B buffer
    extern __shared__ __align__(16) char smem[];
    stage_args(p);
    const int tid = threadIdx.x, lane = tid & 63, wave = tid >> 6;
    half_t *As = reinterpret_cast<half_t *>(smem);   // [2][BM][LD]; AMODE 2: the normalised panel [BM][K + 8]
    const int KP = p.K + 8;                          // panel row (halves): 16 bytes off a multiple of 128, like LD
    half_t *Bs = As + (LNA ? BM * KP : 2 * BM * LD); // [2][BN][LD] or [2][BK][BLD]
    const int wm = wave % WAVES_M, wn = wave / WAVES_M;
    int tm_, tn_;
    tile_of(p, tm_, tn_);
    const int m0 = tm_ * BM, n0 = tn_ * BN;
    const long bz = blockIdx.y;
    const half_t *A = p.A + bz * p.sA;
    const half_t *B = p.B + bz * p.sB;

    // Per-thread global sources; rows and columns past the edge re-read the last
    // valid one (their results are never stored).
    const half_t *ap[PA], *bp[PB];
#pragma unroll
    for (int i = 0; i < PA; i++) { const int c = tid + i * NT; ap[i] = A + (long)min(m0 + (c >> 3), p.M - 1) * p.ldA + (c & 7) * 8; }
#pragma unroll
    for (int i = 0; i < PB; i++) {
        const int c = tid + i * NT;
        if (!B_KN) bp[i] = B + (long)min(n0 + (c >> 3), p.N - 1) * p.ldB + (c & 7) * 8;
        else       bp[i] = B + (long)(c / CPRB) * p.ldB + min(n0 + (c % CPRB) * 8, p.NB - 8);
    }
    // Channels-last gather: a thread's rows are fixed output pixels; (iy0, ix0) is where tap (0, 0) of each lands.
    int aiy0[PA], aix0[PA];
    int atile0 = 0;
    if constexpr (AMODE == 1) {
#pragma unroll
        for (int i = 0; i < PA; i++) {
            const int c = tid + i * NT;
            const int m = min(m0 + (c >> 3), p.M - 1);
            const int pq = p.ag.OH * p.ag.OW;
            const int n = m / pq, rem = m - n * pq, oh = rem / p.ag.OW, ow = rem - oh * p.ag.OW;
            aiy0[i] = oh * p.ag.sy - p.ag.py;
            aix0[i] = ow * p.ag.sx - p.ag.px;
            ap[i] = p.ag.x + (long)n * p.ag.H * p.ag.W * p.ag.C + (c & 7) * 8;
        }
        atile0 = p.ag.split ? (int)bz * (p.K / BK) : 0;
    }
    u32x4 ga[2][PA], gb[2][PB];
    LnfRows<TM> lnf(p, m0 + wm * WTM, lane);
    auto gload = [&](int set, int kt) {
        if constexpr (LNF) lnf.request(p, set, kt);       // (ahead of the tile's own: where those have landed, these have)
        const long ko = (long)kt * BK;
        if constexpr (AMODE == 1) {
            const int t = atile0 + kt, tap = t / p.ag.cpt, ci0 = (t - tap * p.ag.cpt) * BK;       // the same for every lane
            const int kh = tap / p.ag.KW, kw = tap - kh * p.ag.KW;
            const int ddy = kh * p.ag.dy, ddx = kw * p.ag.dx;
#pragma unroll
            for (int i = 0; i < PA; i++) {
                const int iy = aiy0[i] + ddy, ix = aix0[i] + ddx;
                const bool in = (unsigned)iy < (unsigned)p.ag.H && (unsigned)ix < (unsigned)p.ag.W;
                const u32x4 z = {0u, 0u, 0u, 0u};
                ga[set][i] = in ? ldg16(ap[i] + ((long)iy * p.ag.W + ix) * p.ag.C + ci0) : z;
            }
        } else if constexpr (!LNA) {
#pragma unroll
            for (int i = 0; i < PA; i++) ga[set][i] = ldg16(ap[i] + (KTAIL ? min(ko, (long)(p.K - 8 - ((tid + i * NT) & 7) * 8)) : ko));
        }
#pragma unroll
        for (int i = 0; i < PB; i++) {
            const int c = tid + i * NT;
            const long kc = KTAIL ? min(ko, (long)(B_KN ? p.K - 1 - c / CPRB : p.K - 8 - (c & 7) * 8)) : ko;
            gb[set][i] = ldg16(bp[i] + (B_KN ? kc * p.ldB : kc));
        }
    };
    // last: the tile that K ends in (KTAIL)
    const int kleft = p.K - (p.K - 1) / BK * BK;           // 1 .. 64 columns of it
    auto lwrite_a = [&](int set, int buf, bool last) {
        if constexpr (LNA) return;                     // the panel is already there
        if (KTAIL && last) {
#pragma unroll
            for (int i = 0; i < PA; i++) ga[set][i] &= ((tid + i * NT) & 7) * 8 < kleft ? 0xffffffffu : 0u;
        }
#pragma unroll
        for (int i = 0; i < PA; i++) { const int c = tid + i * NT; *reinterpret_cast<u32x4 *>(As + buf * BM * LD + (c >> 3) * LD + (c & 7) * 8) = ga[set][i]; }
    };
    auto lwrite_b = [&](int set, int buf, bool last) {
        if (KTAIL && last) {
#pragma unroll
            for (int i = 0; i < PB; i++) {
                const int c = tid + i * NT;
                gb[set][i] &= (B_KN ? c / CPRB : (c & 7) * 8) < kleft ? 0xffffffffu : 0u;
            }
        }
#pragma unroll
        for (int i = 0; i < PB; i++) {
            const int c = tid + i * NT;
            half_t *dst = !B_KN ? Bs + buf * BSZ + (c >> 3) * LD + (c & 7) * 8 : Bs + buf * BSZ + (c / CPRB) * BLD + (c % CPRB) * 8;
            *reinterpret_cast<u32x4 *>(dst) = gb[set][i];
        }
    };

    float16v acc[TN][TM];
#pragma unroll
    for (int i = 0; i < TN; i++)
#pragma unroll
        for (int j = 0; j < TM; j++)
#pragma unroll
            for (int r = 0; r < 16; r++) acc[i][j][r] = 0.0f;

    const int frow = lane & 31, fk = (lane >> 5) * 8;
    const int aoff = (wm * WTM + frow) * (LNA ? KP : LD) + fk, boff = (wn * WTN + frow) * LD + fk;
    // [K][N] fragments: within each block of 16 lanes, lane i of ds_read_b64_tr_b16
    // receives, for j = 0..3, element i%4 of the 8 bytes addressed by lane 4j + i/4.
    // Pointing lane s at row (k0 + s/4), columns (n0 + 4 (s%4) .. +3) therefore hands
    // lane i the four consecutive k of column n0 + i: the MFMA operand layout.
    const int tboff = (fk + ((lane & 15) >> 2)) * BLD + wn * WTN + ((lane >> 4) & 1) * 16 + (lane & 3) * 4;
    half8v fa[2][TM], fb[2][TN];
    auto fread = [&](int fs, int buf, int ks, int kt) {
        const half_t *as = LNA ? As + aoff + kt * BK + ks * 16 : As + buf * BM * LD + aoff + ks * 16;
        const int jstep = 32 * (LNA ? KP : LD);
#pragma unroll
        for (int j = 0; j < TM; j++) fa[fs][j] = *reinterpret_cast<const half8v *>(as + j * jstep);
        if (!B_KN) {
            const half_t *bs = Bs + buf * BSZ + boff + ks * 16;
#pragma unroll
            for (int i = 0; i < TN; i++) fb[fs][i] = *reinterpret_cast<const half8v *>(bs + i * 32 * LD);
        } else {
            const half_t *bs = Bs + buf * BSZ + tboff + ks * 16 * BLD;
#pragma unroll
            for (int i = 0; i < TN; i++) {
                short4v lo = __builtin_amdgcn_ds_read_tr16_b64_v4i16((__attribute__((address_space(3))) short4v *)(bs + i * 32));
                short4v hi = __builtin_amdgcn_ds_read_tr16_b64_v4i16((__attribute__((address_space(3))) short4v *)(bs + i * 32 + 4 * BLD));
                short8v both = {lo[0], lo[1], lo[2], lo[3], hi[0], hi[1], hi[2], hi[3]};
                fb[fs][i] = __builtin_bit_cast(half8v, both);
            }
        }
    };
    auto mma = [&](int fs) {
#pragma unroll
        for (int i = 0; i < TN; i++)
#pragma unroll
            for (int j = 0; j < TM; j++) acc[i][j] = __builtin_amdgcn_mfma_f32_32x32x16_f16(fb[fs][i], fa[fs][j], acc[i][j], 0, 0, 0);
    };

    const int nk = KTAIL ? (p.K + BK - 1) / BK : p.K / BK;   // the launcher guarantees nk >= 2, and K % 64 == 0 without KTAIL
    gload(0, 0);
    gload(1, 1);
    if constexpr (LNA) {
        // One wave per row, all rows of a wave in flight at once (one trip to memory).  Rows past M repeat the last one.
        constexpr int NW = NT / 64, RB = BM / NW;
        static_assert(RB >= 1 && RB <= 16 && BM % NW == 0, "a wave's rows fit its registers");
        const int e0 = lane * 8;
        const bool mine = e0 < p.K;
        const u32x4 z = {0u, 0u, 0u, 0u};
        const half8v gv = as_half8((p.ln_gamma && mine) ? ldg16(p.ln_gamma + e0) : z);
        const half8v bv = as_half8((p.ln_beta && mine) ? ldg16(p.ln_beta + e0) : z);
        for (int r0 = wave * (BM / NW); r0 < (wave + 1) * (BM / NW); r0 += RB) {
            u32x4 raw[RB];
#pragma unroll
            for (int q = 0; q < RB; q++) raw[q] = mine ? ldg16(A + (long)min(m0 + r0 + q, p.M - 1) * p.ldA + e0) : z;
#pragma unroll
            for (int q = 0; q < RB; q++) {
                const half8v t = as_half8(raw[q]);
                float x[8], sum = 0.0f;
#pragma unroll
                for (int j = 0; j < 8; j++) { x[j] = mine ? (float)t[j] : 0.0f; if (mine) sum += x[j]; }
                sum = wave_sum(sum);
                const float mu = sum / (float)p.K;
                float s2 = 0.0f;
                if (mine) {
#pragma unroll
                    for (int j = 0; j < 8; j++) { const float d = x[j] - mu; s2 = fmaf(d, d, s2); }
                }
                s2 = wave_sum(s2);
                const float rs = 1.0f / sqrtf(s2 / (float)p.K + p.ln_eps);
                if (mine) {
                    half8v o8;
#pragma unroll
                    for (int j = 0; j < 8; j++)
                        o8[j] = ln_norm1(x[j], mu, rs, p.ln_gamma != nullptr, p.ln_gamma ? (float)gv[j] : 0.0f, p.ln_beta != nullptr, p.ln_beta ? (float)bv[j] : 0.0f);
                    *reinterpret_cast<half8v *>(As + (r0 + q) * KP + e0) = o8;
                }
            }
        }
    }
    lwrite_a(0, 0, false);
    lwrite_b(0, 0, false);
    if constexpr (LNF) lnf.template take<true>(0);
    __syncthreads();
    fread(0, 0, 0, 0);

    // MODE 0: steady state; 1: second-to-last tile (nothing left to fetch); 2: last tile.
    // Tile kt is computed from LDS buffer `cur`; register set `gw` holds tile kt+1, set `gl` receives tile kt+2.
    auto body = [&](auto MODE_, int kt, int cur, int gw, int gl) {
        constexpr int MODE = decltype(MODE_)::value;
        constexpr int NM = TM * TN;               // MFMAs per k-step
        constexpr int NR = TM + (B_KN ? 2 * TN : TN);   // fragment reads per k-step
        // Each k-step is pinned to: its fragment reads first, then its MFMAs with the step's
        // memory instructions dealt out between them, so that neither the LDS pipe nor the
        // vector-memory path sees a burst.
        if constexpr (MODE == 0) gload(gl, kt + 2);
        fread(1, cur, 1, kt);
        mma(0);
        __builtin_amdgcn_sched_group_barrier(0x100, NR, 0);
#pragma unroll
        for (int g = 0; g < NM; g++) { __builtin_amdgcn_sched_group_barrier(0x008, 1, 0); __builtin_amdgcn_sched_group_barrier(0x020, (PA + PB + (LNF ? TM : 0) + NM - 1) / NM, 0); }
        __builtin_amdgcn_sched_barrier(0);
        fread(0, cur, 2, kt);
        mma(1);
        if constexpr (MODE < 2) lwrite_a(gw, cur ^ 1, MODE == 1);
        __builtin_amdgcn_sched_group_barrier(0x100, NR, 0);
#pragma unroll
        for (int g = 0; g < NM; g++) { __builtin_amdgcn_sched_group_barrier(0x008, 1, 0); __builtin_amdgcn_sched_group_barrier(0x200, (PA + NM - 1) / NM, 0); }
        __builtin_amdgcn_sched_barrier(0);
        fread(1, cur, 3, kt);
        mma(0);
        if constexpr (MODE < 2) lwrite_b(gw, cur ^ 1, MODE == 1);
        if constexpr (LNF && MODE < 2) lnf.take(gw);
        __builtin_amdgcn_sched_group_barrier(0x100, NR, 0);
#pragma unroll
        for (int g = 0; g < NM; g++) { __builtin_amdgcn_sched_group_barrier(0x008, 1, 0); __builtin_amdgcn_sched_group_barrier(0x200, (PB + NM - 1) / NM, 0); }
        __builtin_amdgcn_sched_barrier(0);
        __syncthreads();
        if constexpr (MODE < 2) fread(0, cur ^ 1, 0, kt + 1);
        mma(1);
        __builtin_amdgcn_sched_group_barrier(0x100, NR, 0);
        __builtin_amdgcn_sched_barrier(0);
    };
    using M0 = std::integral_constant<int, 0>;
    using M1 = std::integral_constant<int, 1>;
    using M2 = std::integral_constant<int, 2>;
    const int npairs = (nk - 2) >> 1;       // steady-state tiles come in (buffer 0, buffer 1) pairs
    int kt = 0;
    for (int pr = 0; pr < npairs; pr++, kt += 2) {
        body(M0{}, kt, 0, 1, 0);
        body(M0{}, kt + 1, 1, 0, 1);
    }
    half4v cb[TN][4] = {};                    // (a folded norm has its bias in biasp)
    ResidualAhead<WTN> res;
    std::conditional_t<LNF, LnFoldRegs<TM, TN>, LnFold<TM>> ln;
    // what the store needs of memory, under the last tile
    auto ends = [&](int kt, int cur, int gw, int gl) __attribute__((always_inline)) {
        body(M1{}, kt, cur, gw, gl);
        if constexpr (LNF) {
            ln.load(p, n0 + wn * WTN, lane, bz);
            lnf.finish(p, ln.r, ln.rmu);
        } else {
            load_col_bias<TN, WTN>(p, cb, n0, wn, lane, bz);
            res.request(p, m0 + wm * WTM, n0 + wn * WTN, lane, bz);
        }
        body(M2{}, kt + 1, cur ^ 1, gl, gw);
    };
    if (nk & 1) {
        body(M0{}, kt, 0, 1, 0);
        ends(kt + 1, 1, 0, 1);
    } else ends(kt, 0, 1, 0);
    __syncthreads();
    store_tile<TM, TN, WTM, WTN, WAVES_M * WAVES_N, 2 * (BM * LD + BSZ) * 2>(p, acc, cb, smem, m0, n0, wm, wn, wave, lane, bz, ln, LNF ? nullptr : &res);
}

template <int BM, int BN, int WM, int WN>
int launch_pipe(GemmArgs a, bool b_kn, int64_t nbatch, hipStream_t st) {
    // the kernel always walks at least two 64-deep tiles (its prologue fetches two ahead): one tile would read past K
    if (a.K <= 64 || a.K % 8) return MI_DECLINE_EXTENT;
    set_tiles(a, BM, BN);
    a.vec_store = rows_vec16(a);
    dim3 grid((unsigned)(a.tiles_m * a.tiles_n), (unsigned)nbatch);
    constexpr int lds = gemm_lds_bytes<BM, BN, 64>();
    if (a.ag.x && a.K % 64) return MI_DECLINE_EXTENT;
    if (a.ag.x) {
        if (b_kn) hipLaunchKernelGGL((gemm_pipe_kernel<BM, BN, WM, WN, 1, 1>), grid, dim3(WM * WN * 64), lds, st, a);
        else      hipLaunchKernelGGL((gemm_pipe_kernel<BM, BN, WM, WN, 0, 1>), grid, dim3(WM * WN * 64), lds, st, a);
    }
    else if (a.K % 64) {
        if (b_kn) hipLaunchKernelGGL((gemm_pipe_kernel<BM, BN, WM, WN, 1, 0, true>), grid, dim3(WM * WN * 64), lds, st, a);
        else      hipLaunchKernelGGL((gemm_pipe_kernel<BM, BN, WM, WN, 0, 0, true>), grid, dim3(WM * WN * 64), lds, st, a);
    }
    else if (a.lnf_stats) {
        if constexpr (BM * BN <= 128 * 128) {
            if (b_kn) hipLaunchKernelGGL((gemm_pipe_kernel<BM, BN, WM, WN, 1, 0, false, true>), grid, dim3(WM * WN * 64), lds, st, a);
            else      hipLaunchKernelGGL((gemm_pipe_kernel<BM, BN, WM, WN, 0, 0, false, true>), grid, dim3(WM * WN * 64), lds, st, a);
        } else return MI_DECLINE_EXTENT;      // the four-wave kernel's tiles
    }
    else if (b_kn) hipLaunchKernelGGL((gemm_pipe_kernel<BM, BN, WM, WN, 1>), grid, dim3(WM * WN * 64), lds, st, a);
    else           hipLaunchKernelGGL((gemm_pipe_kernel<BM, BN, WM, WN, 0>), grid, dim3(WM * WN * 64), lds, st, a);
    return hipGetLastError() == hipSuccess ? MI_OK : MI_ERROR_LAUNCH;
}

template <int BM, int BN, int WM, int WN>
int raise_pipe() {
    constexpr int lds = gemm_lds_bytes<BM, BN, 64>();
    int bad = 0;
    if constexpr (BM * BN <= 128 * 128)
        bad = raise_lds(gemm_pipe_kernel<BM, BN, WM, WN, 0, 0, false, true>, lds) | raise_lds(gemm_pipe_kernel<BM, BN, WM, WN, 1, 0, false, true>, lds);
    return bad | raise_lds(gemm_pipe_kernel<BM, BN, WM, WN, 0>, lds) | raise_lds(gemm_pipe_kernel<BM, BN, WM, WN, 1>, lds) |
           raise_lds(gemm_pipe_kernel<BM, BN, WM, WN, 0, 1>, lds) | raise_lds(gemm_pipe_kernel<BM, BN, WM, WN, 1, 1>, lds) |
           raise_lds(gemm_pipe_kernel<BM, BN, WM, WN, 0, 0, true>, lds) | raise_lds(gemm_pipe_kernel<BM, BN, WM, WN, 1, 0, true>, lds);
}

// The pipelined kernel with the layer norm of A's rows as its prologue (AMODE 2): 64-row tiles, 128 <= K <= 512.
template <int BN, int WM, int WN>
constexpr int lna_lds_bytes(int K) {
    constexpr int kc = BN * (64 + 8), kn = 64 * (BN + 32);
    return (64 * (K + 8) + 2 * (kc > kn ? kc : kn)) * 2;
}
template <int BN, int WM, int WN>
int launch_pipe_ln(GemmArgs a, bool b_kn, hipStream_t st) {
    if (a.K < 128 || a.K % 64 || a.K > MI_LNA_KMAX || a.ag.x) return MI_DECLINE_EXTENT;
    set_tiles(a, 64, BN);
    a.vec_store = rows_vec16(a);
    dim3 grid((unsigned)(a.tiles_m * a.tiles_n), 1);
    const int lds = lna_lds_bytes<BN, WM, WN>(a.K);
    if (b_kn) hipLaunchKernelGGL((gemm_pipe_kernel<64, BN, WM, WN, 1, 2>), grid, dim3(WM * WN * 64), lds, st, a);
    else      hipLaunchKernelGGL((gemm_pipe_kernel<64, BN, WM, WN, 0, 2>), grid, dim3(WM * WN * 64), lds, st, a);
    return hipGetLastError() == hipSuccess ? MI_OK : MI_ERROR_LAUNCH;
}

}  // namespace

int mi_pipe_launch(int tile, const GemmArgs &a, bool b_kn, int64_t nbatch, hipStream_t st) {
    switch (tile) {
        case 0: return launch_pipe<128, 256, 2, 4>(a, b_kn, nbatch, st);
        case 1: return launch_pipe<192, 128, 2, 4>(a, b_kn, nbatch, st);
        case 2: return launch_pipe<128, 128, 2, 4>(a, b_kn, nbatch, st);
        case 3: return launch_pipe<64, 128, 2, 4>(a, b_kn, nbatch, st);
        default: return launch_pipe<64, 64, 2, 2>(a, b_kn, nbatch, st);
    }
}

int mi_pipe_launch_ln(bool wide, const GemmArgs &a, bool b_kn, hipStream_t st) {
    return wide ? launch_pipe_ln<128, 2, 4>(a, b_kn, st) : launch_pipe_ln<64, 2, 2>(a, b_kn, st);
}

int mi_pipe_init() {
    int bad = raise_pipe<128, 256, 2, 4>() | raise_pipe<192, 128, 2, 4>() | raise_pipe<128, 128, 2, 4>() | raise_pipe<64, 128, 2, 4>() | raise_pipe<64, 64, 2, 2>();
    bad |= raise_lds(gemm_pipe_kernel<64, 128, 2, 4, 1, 2>, lna_lds_bytes<128, 2, 4>(MI_LNA_KMAX));
    bad |= raise_lds(gemm_pipe_kernel<64, 128, 2, 4, 0, 2>, lna_lds_bytes<128, 2, 4>(MI_LNA_KMAX));
    bad |= raise_lds(gemm_pipe_kernel<64, 64, 2, 2, 1, 2>, lna_lds_bytes<64, 2, 2>(MI_LNA_KMAX));
    bad |= raise_lds(gemm_pipe_kernel<64, 64, 2, 2, 0, 2>, lna_lds_bytes<64, 2, 2>(MI_LNA_KMAX));
    return bad;
}
