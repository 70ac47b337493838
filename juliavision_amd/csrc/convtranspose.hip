// Transposed convolution for gfx950, in the reference's layout:
//   x (W,H,Cin,N) = [N][Cin][H][W],  w (KW,KH,Cout/g,Cin) = [Cin][Cout/g][KH][KW] (torch's
//   conv_transpose2d weight),  out (OW,OH,Cout,N) = [N][Cout][OH][OW].
// Two routes, as the reference has them (conv.jl:204-294):
//   kernel == stride, no padding / dilation / output padding, one group:
//       every output pixel has exactly one source pixel and one tap, so per image
//           out[co][iy*KH+ky][ix*KW+kx] = w[Cin][(co,ky,kx)]^T . x[Cin][H*W] + bias[co]
//       one GEMM on MFMA whose store does the pixel shuffle.
//   anything else: one thread per output gathers the inputs that reach it (conv.jl:149-191).
#include "common.hpp"

namespace {

struct CtArgs {
    const half_t *x, *w, *bias;
    half_t *out;
    int Wi, Hi, Cin, N, KW, KH, Cout, OW, OH;
    int sx, sy, px, py, dx, dy, groups;
};

// Eight halves of row k at column n0, zero outside [0, K) x [0, N): one 16-byte load at any address, by element at the
// row's end (nothing past the row is read).
__device__ __forceinline__ u32x4 ct_row8(const half_t *base, int k, int K, long N, long n0) {
    u32x4 v = {0u, 0u, 0u, 0u};
    if (k < K) {
        const half_t *p = base + (long)k * N + n0;
        if (n0 + 8 <= N) __builtin_memcpy(&v, p, 16);
        else if (n0 < N) {
            half8v h = as_half8(v);
#pragma unroll
            for (int e = 0; e < 8; e++) if (n0 + e < N) h[e] = p[e];
            v = __builtin_bit_cast(u32x4, h);
        }
    }
    return v;
}

// BM x 64 tile of (co, ky, kx) x pixels, four waves, each 32 pixels x BM / 2 rows.  Both operands have K = Cin as their
// slow axis, so both go to LDS as they lie ([k][columns], 64 channels a stage, the next stage's loads in flight during
// this one's MFMAs) and reach the matrix unit through the transposing LDS read.  A lane ends with four consecutive rows
// of one pixel: for a 2 x 2 kernel the four taps of one output channel, two of them neighbours in an output row, so a
// wave stores 128 contiguous bytes per row.
// Bound by latency at the sizes upsamplers have (256 channels: four trips through memory and LDS).  It replaces a weight
// transpose, a GEMM into scratch and a shuffle pass, three launches: 256 -> 64 channels on 64 x 64 took 11.7 us.
template <int BM, bool TAPS22>
__global__ __launch_bounds__(256) void ct_mfma_kernel(CtArgs a) {
    constexpr int BN = 64, BK = 64, NT = 256, ALD = BM + 32, BLD = BN + 32, TM = BM / 64;
    constexpr int PA = BK * BM / 8 / NT, PB = BK * BN / 8 / NT;
    __shared__ __align__(16) half_t As[2][BK * ALD], Bs[2][BK * BLD];
    const int tid = threadIdx.x, lane = tid & 63, wave = tid >> 6, wm = wave & 1, wn = wave >> 1;
    const int taps = a.KH * a.KW, M = a.Cout * taps;
    const long HW = (long)a.Hi * a.Wi;
    const int m0 = blockIdx.y * BM;
    const long n0 = (long)blockIdx.x * BN;
    const half_t *x = a.x + (long)blockIdx.z * a.Cin * HW;
    u32x4 ra[PA], rb[PB];
    auto load = [&](int k0) {
#pragma unroll
        for (int i = 0; i < PA; i++) { const int c = tid + i * NT; ra[i] = ct_row8(a.w, k0 + c / (BM / 8), a.Cin, M, m0 + c % (BM / 8) * 8); }
#pragma unroll
        for (int i = 0; i < PB; i++) { const int c = tid + i * NT; rb[i] = ct_row8(x, k0 + c / (BN / 8), a.Cin, HW, n0 + c % (BN / 8) * 8); }
    };
    auto put = [&](int buf) {
#pragma unroll
        for (int i = 0; i < PA; i++) { const int c = tid + i * NT; *reinterpret_cast<u32x4 *>(&As[buf][c / (BM / 8) * ALD + c % (BM / 8) * 8]) = ra[i]; }
#pragma unroll
        for (int i = 0; i < PB; i++) { const int c = tid + i * NT; *reinterpret_cast<u32x4 *>(&Bs[buf][c / (BN / 8) * BLD + c % (BN / 8) * 8]) = rb[i]; }
    };
    // transposing read: within each block of 16 lanes lane s points at row k + s / 4, columns 4 (s % 4) .. + 3, and lane i
    // receives four consecutive k of column i
    const int trow = (lane >> 5) * 8 + ((lane & 15) >> 2), tcol = ((lane >> 4) & 1) * 16 + (lane & 3) * 4;
    auto frag = [&](const half_t *s, int ld) {
        const short4v lo = __builtin_amdgcn_ds_read_tr16_b64_v4i16((__attribute__((address_space(3))) short4v *)s);
        const short4v hi = __builtin_amdgcn_ds_read_tr16_b64_v4i16((__attribute__((address_space(3))) short4v *)(s + 4 * ld));
        const short8v both = {lo[0], lo[1], lo[2], lo[3], hi[0], hi[1], hi[2], hi[3]};
        return __builtin_bit_cast(half8v, both);
    };
    float16v acc[TM];
#pragma unroll
    for (int i = 0; i < TM; i++)
#pragma unroll
        for (int r = 0; r < 16; r++) acc[i][r] = 0.0f;
    const int steps = (a.Cin + BK - 1) / BK;
    load(0);
    put(0);
    __syncthreads();
    for (int s = 0; s < steps; s++) {
        if (s + 1 < steps) load((s + 1) * BK);
        const half_t *as = As[s & 1] + trow * ALD + wm * (BM / 2) + tcol, *bs = Bs[s & 1] + trow * BLD + wn * 32 + tcol;
#pragma unroll
        for (int ks = 0; ks < BK / 16; ks++) {
            const half8v fb = frag(bs + ks * 16 * BLD, BLD);
#pragma unroll
            for (int i = 0; i < TM; i++) acc[i] = __builtin_amdgcn_mfma_f32_32x32x16_f16(frag(as + ks * 16 * ALD + i * 32, ALD), fb, acc[i], 0, 0, 0);
        }
        if (s + 1 < steps) put((s + 1) & 1);
        __syncthreads();
    }
    // acc[i][4 g + e] of a lane: row m0 + wm BM / 2 + 32 i + 8 g + 4 (lane / 32) + e, pixel n0 + 32 wn + lane % 32
    const long n = n0 + wn * 32 + (lane & 31);
    if (n >= HW) return;
    const int iy = (int)(n / a.Wi), ix = (int)(n % a.Wi);
    half_t *out = a.out + (long)blockIdx.z * a.Cout * a.OH * a.OW;
#pragma unroll
    for (int i = 0; i < TM; i++)
#pragma unroll
        for (int g = 0; g < 4; g++) {
            const int m = m0 + wm * (BM / 2) + 32 * i + 8 * g + 4 * (lane >> 5);
            if constexpr (TAPS22) {
                if (m < M) {
                    const int co = m >> 2;
                    const float b = a.bias ? (float)a.bias[co] : 0.0f;
                    half_t *dst = out + ((long)co * a.OH + 2 * iy) * a.OW + 2 * ix;
#pragma unroll
                    for (int ky = 0; ky < 2; ky++) {
                        const half2v v = {(half_t)(acc[i][4 * g + 2 * ky] + b), (half_t)(acc[i][4 * g + 2 * ky + 1] + b)};
                        __builtin_memcpy(dst + (long)ky * a.OW, &v, 4);
                    }
                }
            } else {
#pragma unroll
                for (int e = 0; e < 4; e++) {
                    if (m + e < M) {
                        const int co = (m + e) / taps, t = (m + e) - co * taps, ky = t / a.KW, kx = t - ky * a.KW;
                        out[((long)co * a.OH + iy * a.KH + ky) * a.OW + ix * a.KW + kx] = (half_t)(acc[i][4 * g + e] + (a.bias ? (float)a.bias[co] : 0.0f));
                    }
                }
            }
        }
}

// The gather form: the loop order and the fp32 accumulator (seeded with the bias) of the reference's
// convtranspose2d (conv.jl:149-191).
__global__ void ct_gather_kernel(CtArgs a) {
    const long idx = (long)blockIdx.x * blockDim.x + threadIdx.x;
    const long total = (long)a.N * a.Cout * a.OH * a.OW;
    if (idx >= total) return;
    const int ox = (int)(idx % a.OW);
    long t = idx / a.OW;
    const int oy = (int)(t % a.OH); t /= a.OH;
    const int co = (int)(t % a.Cout);
    const int n = (int)(t / a.Cout);
    const int cing = a.Cin / a.groups, coutg = a.Cout / a.groups;
    const int g = co / coutg, cog = co % coutg;
    float acc = a.bias ? (float)a.bias[co] : 0.0f;
    const int bx = ox + a.px, by = oy + a.py;
    for (int ci = g * cing; ci < (g + 1) * cing; ci++) {
        const half_t *xc = a.x + ((long)n * a.Cin + ci) * a.Hi * a.Wi;
        const half_t *wc = a.w + ((long)ci * coutg + cog) * a.KH * a.KW;
        for (int ky = 0; ky < a.KH; ky++) {
            const int ty = by - ky * a.dy;
            if (ty < 0 || ty % a.sy != 0) continue;
            const int iy = ty / a.sy;
            if (iy >= a.Hi) continue;
            for (int kx = 0; kx < a.KW; kx++) {
                const int tx = bx - kx * a.dx;
                if (tx < 0 || tx % a.sx != 0) continue;
                const int ix = tx / a.sx;
                if (ix >= a.Wi) continue;
                acc = fmaf((float)xc[iy * a.Wi + ix], (float)wc[ky * a.KW + kx], acc);
            }
        }
    }
    a.out[idx] = (half_t)acc;
}

int fill(CtArgs &a, void *out, const void *x, const void *w, const void *bias,
         int64_t Wi, int64_t Hi, int64_t Cin, int64_t N, int64_t KW, int64_t KH, int64_t Cout,
         int64_t sx, int64_t sy, int64_t px, int64_t py, int64_t dx, int64_t dy, int64_t opx, int64_t opy, int64_t groups) {
    if (Wi < 1 || Hi < 1 || Cin < 1 || N < 0 || KW < 1 || KH < 1 || Cout < 1) return MI_DECLINE_EXTENT;
    if (sx < 1 || sy < 1 || dx < 1 || dy < 1 || px < 0 || py < 0 || opx < 0 || opy < 0 || groups < 1) return MI_DECLINE_EXTENT;
    if (Cin % groups || Cout % groups) return MI_DECLINE_EXTENT;
    // ATen's rule: the output padding fills the gap a stride (or dilation) leaves, no more
    if ((opx >= sx && opx >= dx) || (opy >= sy && opy >= dy)) return MI_DECLINE_EXTENT;
    const int64_t OW = mi_convtransposesize(Wi, KW, sx, px, dx, opx), OH = mi_convtransposesize(Hi, KH, sy, py, dy, opy);
    if (OW < 1 || OH < 1) return MI_DECLINE_EXTENT;
    if (Wi * Hi * Cin > INT32_MAX || OW * OH * Cout > INT32_MAX || Cin * (Cout / groups) * KW * KH > INT32_MAX || N > 65535) return MI_DECLINE_EXTENT;
    a.x = (const half_t *)x; a.w = (const half_t *)w; a.bias = (const half_t *)bias; a.out = (half_t *)out;
    a.Wi = (int)Wi; a.Hi = (int)Hi; a.Cin = (int)Cin; a.N = (int)N; a.KW = (int)KW; a.KH = (int)KH; a.Cout = (int)Cout;
    a.OW = (int)OW; a.OH = (int)OH;
    a.sx = (int)sx; a.sy = (int)sy; a.px = (int)px; a.py = (int)py; a.dx = (int)dx; a.dy = (int)dy; a.groups = (int)groups;
    return MI_OK;
}

// shufflecase, conv.jl:204-209; the output padding is zero by the caller's check
bool shuffle_ok(const CtArgs &a, int64_t opx, int64_t opy) {
    return a.groups == 1 && a.px == 0 && a.py == 0 && a.dx == 1 && a.dy == 1 && opx == 0 && opy == 0 && a.KW == a.sx && a.KH == a.sy;
}

template <int BM>
int launch_ct(const CtArgs &a, hipStream_t st) {
    const int64_t M = (int64_t)a.Cout * a.KH * a.KW, HW = (int64_t)a.Hi * a.Wi;
    const dim3 grid((unsigned)ceil_div(HW, 64), (unsigned)ceil_div(M, BM), (unsigned)a.N);
    if (ceil_div(M, BM) > 65535) return MI_DECLINE_EXTENT;
    if (a.KW == 2 && a.KH == 2) hipLaunchKernelGGL((ct_mfma_kernel<BM, true>), grid, dim3(256), 0, st, a);
    else                        hipLaunchKernelGGL((ct_mfma_kernel<BM, false>), grid, dim3(256), 0, st, a);
    return hipGetLastError() == hipSuccess ? MI_OK : MI_ERROR_LAUNCH;
}

}  // namespace

extern "C" {

int64_t mi_convtransposesize(int64_t n, int64_t k, int64_t s, int64_t p, int64_t d, int64_t op) {
    return (n - 1) * s - 2 * p + d * (k - 1) + op + 1;
}

int mi_convtranspose2d_f16_plan(int64_t Wi, int64_t Hi, int64_t Cin, int64_t N, int64_t KW, int64_t KH, int64_t Cout,
                                int64_t sx, int64_t sy, int64_t px, int64_t py, int64_t dx, int64_t dy,
                                int64_t opx, int64_t opy, int64_t groups) {
    CtArgs a;
    if (fill(a, nullptr, nullptr, nullptr, nullptr, Wi, Hi, Cin, N, KW, KH, Cout, sx, sy, px, py, dx, dy, opx, opy, groups) != MI_OK)
        return MI_CONVT_DECLINE;
    return shuffle_ok(a, opx, opy) ? MI_CONVT_GEMM_SHUFFLE : MI_CONVT_GATHER;
}

size_t mi_convtranspose2d_f16_workspace(int64_t Wi, int64_t Hi, int64_t Cin, int64_t N, int64_t KW, int64_t KH, int64_t Cout,
                                        int64_t sx, int64_t sy, int64_t px, int64_t py, int64_t dx, int64_t dy,
                                        int64_t opx, int64_t opy, int64_t groups) {
    CtArgs a;
    if (fill(a, nullptr, nullptr, nullptr, nullptr, Wi, Hi, Cin, N, KW, KH, Cout, sx, sy, px, py, dx, dy, opx, opy, groups) != MI_OK) return 0;
    if (!shuffle_ok(a, opx, opy)) return 0;
    // Nothing is written there: both kernels work in registers and LDS.  The answer stays what a weight transpose, an expanded
    // bias and an unshuffled result would take, which callers have sized their buffers by.
    const int64_t M = (int64_t)a.Cout * a.KH * a.KW, HW = (int64_t)a.Hi * a.Wi;
    return round_up((size_t)M * a.Cin * 2, 256) + round_up((size_t)M * 2, 256) + round_up((size_t)a.N * M * HW * 2, 256) +
           mi_internal_gemm_workspace(M, a.Cin, HW, a.N);
}

int mi_convtranspose2d_f16(void *out, const void *x, const void *w, const void *bias,
                           int64_t Wi, int64_t Hi, int64_t Cin, int64_t N, int64_t KW, int64_t KH, int64_t Cout,
                           int64_t sx, int64_t sy, int64_t px, int64_t py, int64_t dx, int64_t dy,
                           int64_t opx, int64_t opy, int64_t groups, void *ws, size_t ws_bytes, void *stream) {
    if (!mi_ready()) return MI_ERROR_DEVICE;
    if (!out || !x || !w) return MI_DECLINE_OPERANDS;
    CtArgs a;
    int rc = fill(a, out, x, w, bias, Wi, Hi, Cin, N, KW, KH, Cout, sx, sy, px, py, dx, dy, opx, opy, groups);
    if (rc != MI_OK) return rc;
    if (N == 0) return MI_OK;
    hipStream_t st = (hipStream_t)stream;
    if (!shuffle_ok(a, opx, opy)) {
        const long total = (long)a.N * a.Cout * a.OH * a.OW;
        if (ceil_div(total, 256) > INT32_MAX) return MI_DECLINE_EXTENT;
        hipLaunchKernelGGL(ct_gather_kernel, dim3((unsigned)ceil_div(total, 256)), dim3(256), 0, st, a);
        return hipGetLastError() == hipSuccess ? MI_OK : MI_ERROR_LAUNCH;
    }
    // 128 rows a tile once that still gives every CU two workgroups, else 64
    const int64_t wide = ceil_div((int64_t)a.Hi * a.Wi, 64) * ceil_div((int64_t)a.Cout * a.KH * a.KW, 128) * a.N;
    return wide >= 2 * (int64_t)mi_num_cus() ? launch_ct<128>(a, st) : launch_ct<64>(a, st);
}

}  // extern "C"
