// fp16 GEMM for gfx950, the tiled kernel for what the others do not take: extents, pitches and addresses that are not
// multiples of eight halves (a 51865-word vocabulary, an odd head count, a sliced operand), and K <= 64.
#include "gemm_common.hpp"

namespace {

// Eight halves of a row from column k0, zero from column K on.  ALIGNED: K % 8 == 0 and 16-byte addresses; otherwise the
// load is still one 16-byte instruction (the target takes any address) except at the row's end, which is read by element:
// nothing past the row is touched.
template <bool ALIGNED>
__device__ __forceinline__ u32x4 row8(const half_t *row, int k0, int K) {
    u32x4 v = {0u, 0u, 0u, 0u};
    if (k0 + 8 <= K) {
        if constexpr (ALIGNED) v = ldg16(row + k0);
        else __builtin_memcpy(&v, row + k0, 16);
    } else if (!ALIGNED && k0 < K) {
        half8v h = as_half8(v);
#pragma unroll
        for (int e = 0; e < 8; e++) if (k0 + e < K) h[e] = row[k0 + e];
        v = __builtin_bit_cast(u32x4, h);
    }
    return v;
}

// BM x BN output tile, KG groups of four waves (2 x 2 sub-tiles each) that take every KG-th 64-deep tile of K and sum
// their accumulators through LDS at the end.  Bound by latency: such calls are small (their rows cannot be moved in
// aligned 16-byte pieces, so nobody lays out a large one that way on purpose).  The next tile's loads are in flight
// during this tile's MFMAs.  A call with few output tiles and a long K is a serial chain of K / 64 trips through memory,
// LDS and a barrier: KG = 4 cuts the chain, not the work.
// Against the kernel with one thread per output that stood here: 2 x 464 -> 73 44.4 us, 3 x 311 -> 106 31.1 us before.
template <int BM, int BN, int KG, bool B_KN, bool ALIGNED>
__global__ __launch_bounds__(256 * KG) void gemm_any_kernel(GemmArgs p) {
    constexpr int NT = 256, BK = 64, LD = BK + 8;
    constexpr int WTM = BM / 2, WTN = BN / 2, TM = WTM / 32, TN = WTN / 32;
    constexpr int PA = BM * 8 / NT, PB = BN * 8 / NT;
    constexpr int GROUP = 2 * (BM + BN) * LD;               // halves of one group's double buffer
    extern __shared__ __align__(16) char smem[];
    stage_args(p);
    const int tid = threadIdx.x & 255, group = threadIdx.x >> 8, lane = tid & 63, wave = tid >> 6;
    half_t *As = reinterpret_cast<half_t *>(smem) + group * GROUP, *Bs = As + 2 * BM * LD;
    const int wm = wave & 1, wn = wave >> 1;
    int tm_, tn_;
    tile_of(p, tm_, tn_);
    const int m0 = tm_ * BM, n0 = tn_ * BN;
    const long bz = blockIdx.y;
    const half_t *A = p.A + bz * p.sA, *B = p.B + bz * p.sB;

    u32x4 ra[PA], rb[PB], rn[8];
    // [K][N]: a thread moves an 8 (k) x 8 (n) block, transposed on its way into LDS; a tile has BN such blocks
    const bool mine = tid < BN;
    auto load = [&](int kt) {
        const int k0 = kt * BK;
#pragma unroll
        for (int i = 0; i < PA; i++) {
            const int c = tid + i * NT;
            ra[i] = row8<ALIGNED>(A + (long)min(m0 + (c >> 3), p.M - 1) * p.ldA, k0 + (c & 7) * 8, p.K);
        }
        if constexpr (B_KN) {
#pragma unroll
            for (int j = 0; j < 8; j++) {
                const int k = k0 + (tid & 7) * 8 + j;
                const u32x4 z = {0u, 0u, 0u, 0u};
                rn[j] = mine && k < p.K ? row8<ALIGNED>(B + (long)k * p.ldB, n0 + (tid >> 3) * 8, p.NB) : z;
            }
        } else {
#pragma unroll
            for (int i = 0; i < PB; i++) {
                const int c = tid + i * NT;
                rb[i] = row8<ALIGNED>(B + (long)min(n0 + (c >> 3), p.N - 1) * p.ldB, k0 + (c & 7) * 8, p.K);
            }
        }
    };
    auto put = [&](int buf) {
#pragma unroll
        for (int i = 0; i < PA; i++) { const int c = tid + i * NT; *reinterpret_cast<u32x4 *>(As + buf * BM * LD + (c >> 3) * LD + (c & 7) * 8) = ra[i]; }
        half_t *bs = Bs + buf * BN * LD;
        if constexpr (B_KN) {
            if (mine) {
#pragma unroll
                for (int w = 0; w < 4; w++) {               // dword w of each row holds columns 2w, 2w+1
                    u32x4 lo, hi;
#pragma unroll
                    for (int q = 0; q < 4; q++) { lo[q] = pack_lo(rn[2 * q][w], rn[2 * q + 1][w]); hi[q] = pack_hi(rn[2 * q][w], rn[2 * q + 1][w]); }
                    half_t *dst = bs + ((tid >> 3) * 8 + 2 * w) * LD + (tid & 7) * 8;
                    *reinterpret_cast<u32x4 *>(dst) = lo;
                    *reinterpret_cast<u32x4 *>(dst + LD) = hi;
                }
            }
        } else {
#pragma unroll
            for (int i = 0; i < PB; i++) { const int c = tid + i * NT; *reinterpret_cast<u32x4 *>(bs + (c >> 3) * LD + (c & 7) * 8) = rb[i]; }
        }
    };

    float16v acc[TN][TM];
#pragma unroll
    for (int i = 0; i < TN; i++)
#pragma unroll
        for (int j = 0; j < TM; j++)
#pragma unroll
            for (int r = 0; r < 16; r++) acc[i][j][r] = 0.0f;

    const int nk = (p.K + BK - 1) / BK, steps = (nk + KG - 1) / KG;      // every group takes the same number of steps: tiles past K are zeros
    load(group);
    put(0);
    __syncthreads();
    const int frow = lane & 31, fk = (lane >> 5) * 8;
    for (int s = 0; s < steps; s++) {
        const bool more = s + 1 < steps;
        if (more) load((s + 1) * KG + group);
        const half_t *as = As + (s & 1) * BM * LD + (wm * WTM + frow) * LD + fk;
        const half_t *bs = Bs + (s & 1) * BN * LD + (wn * WTN + frow) * LD + fk;
#pragma unroll
        for (int ks = 0; ks < BK / 16; ks++) {
            half8v fa[TM], fb[TN];
#pragma unroll
            for (int j = 0; j < TM; j++) fa[j] = *reinterpret_cast<const half8v *>(as + j * 32 * LD + ks * 16);
#pragma unroll
            for (int i = 0; i < TN; i++) fb[i] = *reinterpret_cast<const half8v *>(bs + i * 32 * LD + ks * 16);
#pragma unroll
            for (int i = 0; i < TN; i++)
#pragma unroll
                for (int j = 0; j < TM; j++) acc[i][j] = __builtin_amdgcn_mfma_f32_32x32x16_f16(fb[i], fa[j], acc[i][j], 0, 0, 0);
        }
        if (more) put((s + 1) & 1);
        __syncthreads();
    }
    if constexpr (KG > 1) {
        // groups 1 .. KG - 1 leave their accumulators in LDS, group 0 adds them in that order and stores
        static_assert(TM == 1 && TN == 1, "one accumulator tile a wave");
        float *part = reinterpret_cast<float *>(smem);
        if (group > 0) {
#pragma unroll
            for (int r = 0; r < 16; r++) part[((group - 1) * 16 + r) * NT + tid] = acc[0][0][r];
        }
        __syncthreads();
        if (group > 0) return;
#pragma unroll
        for (int g = 0; g < KG - 1; g++)
#pragma unroll
            for (int r = 0; r < 16; r++) acc[0][0][r] += part[(g * 16 + r) * NT + tid];
        asm volatile("s_waitcnt lgkmcnt(0)" ::: "memory");
        // the store's staging must not overrun sums that a slower wave of this group still reads: it lies behind them
    }
    half4v cb[TN][4];
    load_col_bias<TN, WTN>(p, cb, n0, wn, lane, bz);
    char *stage = KG > 1 ? smem + (KG - 1) * 16 * NT * 4 : smem;
    store_tile<TM, TN, WTM, WTN, 4, 2 * (BM + BN) * LD * 2>(p, acc, cb, stage, m0, n0, wm, wn, wave, lane, bz);
}

template <int BM, int BN, int KG>
constexpr int any_lds_bytes() { return KG * 2 * (BM + BN) * 72 * 2; }

template <int BM, int BN, int KG, bool ALIGNED>
int launch_any(GemmArgs a, bool b_kn, int64_t nbatch, hipStream_t st) {
    set_tiles(a, BM, BN);
    a.vec_store = rows_vec16(a);
    dim3 grid((unsigned)(a.tiles_m * a.tiles_n), (unsigned)nbatch);
    constexpr int lds = any_lds_bytes<BM, BN, KG>();
    if (b_kn) hipLaunchKernelGGL((gemm_any_kernel<BM, BN, KG, true, ALIGNED>), grid, dim3(256 * KG), lds, st, a);
    else      hipLaunchKernelGGL((gemm_any_kernel<BM, BN, KG, false, ALIGNED>), grid, dim3(256 * KG), lds, st, a);
    return hipGetLastError() == hipSuccess ? MI_OK : MI_ERROR_LAUNCH;
}

}  // namespace

// `addressable`: K % 8 == 0 and 16-byte rows (only K <= 64 comes here then).  128 x 128 tiles once they give every CU
// one; with 64 x 64 tiles below half a chip and more than four tiles of K, the K-groups.
int mi_any_launch(const GemmArgs &a, bool b_kn, bool addressable, int64_t nbatch, hipStream_t st) {
    if (addressable) return launch_any<64, 64, 1, true>(a, b_kn, nbatch, st);
    const int64_t big = ceil_div(a.M, 128) * ceil_div(a.N, 128) * nbatch, small = ceil_div(a.M, 64) * ceil_div(a.N, 64) * nbatch;
    if (big >= mi_num_cus()) return launch_any<128, 128, 1, false>(a, b_kn, nbatch, st);
    if (small <= mi_num_cus() / 2 && a.K > 256) return launch_any<64, 64, 4, false>(a, b_kn, nbatch, st);
    return launch_any<64, 64, 1, false>(a, b_kn, nbatch, st);
}

int mi_any_init() {
    int bad = 0;
    bad |= raise_lds(gemm_any_kernel<64, 64, 4, true, false>, any_lds_bytes<64, 64, 4>());
    bad |= raise_lds(gemm_any_kernel<64, 64, 4, false, false>, any_lds_bytes<64, 64, 4>());
    bad |= raise_lds(gemm_any_kernel<128, 128, 1, true, false>, any_lds_bytes<128, 128, 1>());
    bad |= raise_lds(gemm_any_kernel<128, 128, 1, false, false>, any_lds_bytes<128, 128, 1>());
    return bad;
}
