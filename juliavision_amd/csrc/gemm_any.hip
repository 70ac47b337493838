// fp16 GEMM for gfx950, the tiled kernel for what the others do not take: extents, pitches and addresses that are not
// multiples of eight halves (a 51865-word vocabulary, an odd head count, a sliced operand), and K <= 64.
#include "gemm_common.hpp"

namespace {

// Eight halves of a row of `len` around column c, in one 16-byte load (the target takes any address): where they would run past
// the row, the row's last eight.  place_row8 puts them where they belong when they are needed, not when they are asked for: a
// load by element there cost its column of tiles eight trips to memory a row (35 x 4743 -> 723 121 us).
// Rows shorter than eight are read by element, by instances of their own (SHORT): a branch around the load would end in a copy
// of its result, which waits for it.  For the same reason an element past the row is the row's last one, and cleared in its place.
enum RowLoad { ALIGNED, ANY, SHORT };
template <RowLoad ROW>
__device__ __forceinline__ u32x4 load_row8(const half_t *row, int c, int len) {
    u32x4 v = {0u, 0u, 0u, 0u};
    if constexpr (ROW == ALIGNED) v = ldg16(row + min(c, len - 8));
    else if constexpr (ROW == ANY) __builtin_memcpy(&v, row + min(c, len - 8), 16);
    else {
        half8v h;
#pragma unroll
        for (int e = 0; e < 8; e++) h[e] = row[min(c + e, len - 1)];
        v = __builtin_bit_cast(u32x4, h);
    }
    return v;
}
// Columns c .. c + 7 of what load_row8 brought, zeros from column len on.
template <RowLoad ROW>
__device__ __forceinline__ u32x4 place_row8(u32x4 v, int c, int len) {
    if constexpr (ROW == SHORT) {                         // in place already
        half8v h = as_half8(v);
#pragma unroll
        for (int e = 0; e < 8; e++) h[e] = c + e < len ? h[e] : (half_t)0.0f;
        return __builtin_bit_cast(u32x4, h);
    }
    const uint32_t by = (uint32_t)min(max(c + 8 - len, 0), 8);                      // halves to drop
    const uint32_t two = by & 2 ? ~0u : 0u, four = by & 4 ? ~0u : 0u, keep = by & 8 ? 0u : ~0u;
    const auto pick = [](uint32_t m, uint32_t a, uint32_t b) { return (a & m) | (b & ~m); };
    uint32_t x0 = v[0] & keep, x1 = v[1] & keep, x2 = v[2] & keep, x3 = v[3] & keep;
    x0 = pick(four, x2, x0); x1 = pick(four, x3, x1); x2 &= ~four; x3 &= ~four;
    x0 = pick(two, x1, x0); x1 = pick(two, x2, x1); x2 = pick(two, x3, x2); x3 &= ~two;
    const uint32_t one = (by & 1) * 16;
    const u32x4 r = {__builtin_amdgcn_alignbit(x1, x0, one), __builtin_amdgcn_alignbit(x2, x1, one), __builtin_amdgcn_alignbit(x3, x2, one), x3 >> one};
    return r;
}

// BM x BN output tile, KG groups of four waves (2 x 2 sub-tiles each) that take every KG-th 64-deep tile of K and sum
// their accumulators through LDS at the end.  Bound by latency: such calls are small (their rows cannot be moved in
// aligned 16-byte pieces, so nobody lays out a large one that way on purpose).  A tile's loads have two tiles' time to arrive, in two
// register sets.  A call with few output tiles and a long K is a serial chain of K / 64 trips through memory, LDS and a barrier:
// KG = 4 cuts the chain, not the work.  The [K][N] operand keeps its layout in LDS and is read with ds_read_b64_tr_b16; it was
// transposed in registers by a quarter of the threads.  us, before -> now: 45 x 3553 -> 1292 81 -> 21, 3593 x 376 -> 197 31 -> 8.4,
// 10 x 252 -> 132 19 -> 5.2, 1500 x 1283 -> 1281 66 -> 21, 2237 x 1000 -> 2437 108 -> 33 ([K][N] weights); 35 x 4743 -> 723 39 -> 26,
// 164 x 190 -> 287 7.4 -> 4.8, 1500 x 1283 -> 1281 22.5 -> 19.8, 2237 x 1001 -> 2437 32.7 -> 33.3 ([N][K]).
template <int BM, int BN, int KG, bool B_KN, RowLoad ROW_A, RowLoad ROW_B>
__global__ __launch_bounds__(256 * KG) void gemm_any_kernel(GemmArgs p) {
    constexpr int NT = 256, BK = 64, LD = BK + 8;
    constexpr bool ONE = ROW_A == SHORT;                    // K < 8: a single tile
    constexpr int WTM = BM / 2, WTN = BN / 2, TM = WTM / 32, TN = WTN / 32;
    constexpr int PA = BM * 8 / NT, PB = BN * 8 / NT;
    constexpr int BLD = BN + 8, CPRB = BN / 8;              // [K][N]: halves and chunks of a k-row
    constexpr int BSZ = B_KN ? BK * BLD : BN * LD, GROUP = 2 * (BM * LD + BSZ);      // halves of one group's double buffer
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

    u32x4 ra[2][PA], rb[2][PB];
    auto load = [&](auto SET, int kt) {
        constexpr int set = decltype(SET)::value;
        const int k0 = kt * BK;
#pragma unroll
        for (int i = 0; i < PA; i++) {
            const int c = tid + i * NT;
            ra[set][i] = load_row8<ROW_A>(A + (long)min(m0 + (c >> 3), p.M - 1) * p.ldA, k0 + (c & 7) * 8, p.K);
        }
#pragma unroll
        for (int i = 0; i < PB; i++) {
            const int c = tid + i * NT;
            if constexpr (B_KN) rb[set][i] = load_row8<ROW_B>(B + (long)min(k0 + c / CPRB, p.K - 1) * p.ldB, n0 + (c % CPRB) * 8, p.NB);
            else rb[set][i] = load_row8<ROW_B>(B + (long)min(n0 + (c >> 3), p.N - 1) * p.ldB, k0 + (c & 7) * 8, p.K);
        }
    };
    auto put = [&](auto SET, int kt) {
        constexpr int set = decltype(SET)::value;
        const int k0 = kt * BK;
        if (k0 + BK > p.K) {                                // uniform: the tile that K ends in, or one past it
#pragma unroll
            for (int i = 0; i < PA; i++) ra[set][i] = place_row8<ROW_A>(ra[set][i], k0 + ((tid + i * NT) & 7) * 8, p.K);
#pragma unroll
            for (int i = 0; i < PB; i++) {
                if constexpr (B_KN) rb[set][i] &= k0 + (tid + i * NT) / CPRB < p.K ? 0xffffffffu : 0u;
                else rb[set][i] = place_row8<ROW_B>(rb[set][i], k0 + ((tid + i * NT) & 7) * 8, p.K);
            }
        }
        if (B_KN && n0 + BN > p.NB) {                       // uniform: the column tile that the rows end in
#pragma unroll
            for (int i = 0; i < PB; i++) rb[set][i] = place_row8<ROW_B>(rb[set][i], n0 + ((tid + i * NT) % CPRB) * 8, p.NB);
        }
#pragma unroll
        for (int i = 0; i < PA; i++) { const int c = tid + i * NT; *reinterpret_cast<u32x4 *>(As + set * BM * LD + (c >> 3) * LD + (c & 7) * 8) = ra[set][i]; }
#pragma unroll
        for (int i = 0; i < PB; i++) {
            const int c = tid + i * NT;
            *reinterpret_cast<u32x4 *>(Bs + set * BSZ + (B_KN ? (c / CPRB) * BLD + (c % CPRB) * 8 : (c >> 3) * LD + (c & 7) * 8)) = rb[set][i];
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
    const int frow = lane & 31, fk = (lane >> 5) * 8;
    const int tboff = (fk + ((lane & 15) >> 2)) * BLD + wn * WTN + ((lane >> 4) & 1) * 16 + (lane & 3) * 4;
    using I0 = std::integral_constant<int, 0>;
    using I1 = std::integral_constant<int, 1>;
    load(I0{}, group);
    if constexpr (!ONE) load(I1{}, KG + group);
    put(I0{}, group);
    __syncthreads();
    // step s: tile s KG + group lies in buffer CUR, its successor is on its way in the other set.  What is asked for past the last tile
    // lies inside the rows: behind a condition the compiler would wait for all loads at every step.
    auto step = [&](auto CUR, int s) {
        constexpr int cur = decltype(CUR)::value;
        if constexpr (!ONE) load(CUR, (s + 2) * KG + group);
        const half_t *as = As + cur * BM * LD + (wm * WTM + frow) * LD + fk;
#pragma unroll
        for (int ks = 0; ks < BK / 16; ks++) {
            half8v fa[TM], fb[TN];
#pragma unroll
            for (int j = 0; j < TM; j++) fa[j] = *reinterpret_cast<const half8v *>(as + j * 32 * LD + ks * 16);
#pragma unroll
            for (int i = 0; i < TN; i++) {
                if constexpr (B_KN) {
                    const half_t *bs = Bs + cur * BSZ + tboff + ks * 16 * BLD + i * 32;
                    const short4v lo = __builtin_amdgcn_ds_read_tr16_b64_v4i16((__attribute__((address_space(3))) short4v *)bs);
                    const short4v hi = __builtin_amdgcn_ds_read_tr16_b64_v4i16((__attribute__((address_space(3))) short4v *)(bs + 4 * BLD));
                    const short8v both = {lo[0], lo[1], lo[2], lo[3], hi[0], hi[1], hi[2], hi[3]};
                    fb[i] = __builtin_bit_cast(half8v, both);
                } else fb[i] = *reinterpret_cast<const half8v *>(Bs + cur * BSZ + (wn * WTN + frow + i * 32) * LD + fk + ks * 16);
            }
#pragma unroll
            for (int i = 0; i < TN; i++)
#pragma unroll
                for (int j = 0; j < TM; j++) acc[i][j] = __builtin_amdgcn_mfma_f32_32x32x16_f16(fb[i], fa[j], acc[i][j], 0, 0, 0);
        }
    };
    if constexpr (ONE) step(I0{}, 0);
    else {
        for (int s = 0;; s += 2) {
            step(I0{}, s);
            if (s + 1 >= steps) break;
            put(I1{}, (s + 1) * KG + group);
            __syncthreads();
            step(I1{}, s + 1);
            if (s + 2 >= steps) break;
            put(I0{}, (s + 2) * KG + group);
            __syncthreads();
        }
    }
    __syncthreads();
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
    store_tile<TM, TN, WTM, WTN, 4, GROUP * 2>(p, acc, cb, stage, m0, n0, wm, wn, wave, lane, bz);
}

template <int BM, int BN, int KG>
constexpr int any_lds_bytes() {                             // either layout of B
    constexpr int nk = BN * 72, kn = 64 * (BN + 8);
    return KG * 2 * (BM * 72 + (nk > kn ? nk : kn)) * 2;
}

template <int BM, int BN, int KG, bool B_KN, RowLoad ROW_A, RowLoad ROW_B = ROW_A>
int launch_any(GemmArgs a, int64_t nbatch, hipStream_t st) {
    set_tiles(a, BM, BN);
    a.vec_store = rows_vec16(a);
    const dim3 grid((unsigned)(a.tiles_m * a.tiles_n), (unsigned)nbatch);
    hipLaunchKernelGGL((gemm_any_kernel<BM, BN, KG, B_KN, ROW_A, ROW_B>), grid, dim3(256 * KG), (any_lds_bytes<BM, BN, KG>()), st, a);
    return hipGetLastError() == hipSuccess ? MI_OK : MI_ERROR_LAUNCH;
}
template <int BM, int BN, int KG, RowLoad ROW>
int launch_any(const GemmArgs &a, bool b_kn, int64_t nbatch, hipStream_t st) {
    return b_kn ? launch_any<BM, BN, KG, true, ROW>(a, nbatch, st) : launch_any<BM, BN, KG, false, ROW>(a, nbatch, st);
}

}  // namespace

// `addressable`: K % 8 == 0 and 16-byte rows (only K <= 64 comes here then).  128 x 128 tiles once they give every CU
// one; with 64 x 64 tiles below half a chip and more than four tiles of K, the K-groups.
int mi_any_launch(const GemmArgs &a, bool b_kn, bool addressable, int64_t nbatch, hipStream_t st) {
    if (addressable) return launch_any<64, 64, 1, ALIGNED>(a, b_kn, nbatch, st);
    // rows shorter than a load: of A (and of a K-contiguous B) where K < 8 -- a 1 x 1 convolution of an image's three channels, 6.6 us
    // by element as the whole of B was, 4.2 with B in wide loads --, of a [K][N] operand where N < 8
    if (a.K < 8) {
        if (!b_kn) return launch_any<64, 64, 1, false, SHORT>(a, nbatch, st);
        return a.NB < 8 ? launch_any<64, 64, 1, true, SHORT>(a, nbatch, st) : launch_any<64, 64, 1, true, SHORT, ANY>(a, nbatch, st);
    }
    if (b_kn && a.NB < 8) return launch_any<64, 64, 1, true, ANY, SHORT>(a, nbatch, st);
    const int64_t big = ceil_div(a.M, 128) * ceil_div(a.N, 128) * nbatch, small = ceil_div(a.M, 64) * ceil_div(a.N, 64) * nbatch;
    if (big >= mi_num_cus()) return launch_any<128, 128, 1, ANY>(a, b_kn, nbatch, st);
    if (small <= mi_num_cus() / 2 && a.K > 256) return launch_any<64, 64, 4, ANY>(a, b_kn, nbatch, st);
    return launch_any<64, 64, 1, ANY>(a, b_kn, nbatch, st);
}

int mi_any_init() {
    int bad = 0;
    bad |= raise_lds(gemm_any_kernel<64, 64, 4, true, ANY, ANY>, any_lds_bytes<64, 64, 4>());
    bad |= raise_lds(gemm_any_kernel<64, 64, 4, false, ANY, ANY>, any_lds_bytes<64, 64, 4>());
    bad |= raise_lds(gemm_any_kernel<128, 128, 1, true, ANY, ANY>, any_lds_bytes<128, 128, 1>());
    bad |= raise_lds(gemm_any_kernel<128, 128, 1, false, ANY, ANY>, any_lds_bytes<128, 128, 1>());
    return bad;
}
