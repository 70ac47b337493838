// fp16 GEMM for gfx950, decode-sized: up to eight rows of activations against weights of either layout, with a layer norm of the
// rows in front or without.
#include "gemm_common.hpp"

namespace {

// Decode-sized M (<= 8): bandwidth- and latency-bound.  Every weight byte is read once with
// 16-byte loads, a thread's loads are all issued before the first is used, and the activations
// (a few KB) are staged in LDS.  Products go through v_dot2_f32_f16: fp16 pairs, fp32 sum.
//
// [K][F] weights: a thread owns 8 consecutive columns, 16 threads span 128 columns, the 16 thread
// rows of a workgroup take interleaved k-pairs.  K is split over workgroups so that the whole chip
// pulls on HBM; each split writes an fp32 partial plane and skinny_epilogue_kernel sums the planes
// (the reference's split-K planes + mm_epilogue_kernel!, matmul.jl:192-217).
// Layer-norm statistics of up to MT rows of A, one wave per row, in the summation order of
// layernorm_vec_kernel (a lane takes the 16-byte chunks lane, lane + 64, ...; butterfly over the wave):
// the fused result is bit-identical to running that kernel first.  stats[m] = (mean, rstd).
template <int MT, int NCH = 8, int NWAVES = 4>              // rows up to NCH * 512 halves stay in registers between the passes
__device__ __forceinline__ void ln_row_stats(const GemmArgs &p, float (*stats)[2], int tid) {
    const int lane = tid & 63, wave = tid >> 6;
    for (int m = wave; m < MT && m < p.M; m += NWAVES) {
        const half_t *row = p.A + (long)m * p.ldA;
        float s = 0.0f, s2 = 0.0f;
        if (p.K <= NCH * 512) {
            u32x4 raw[NCH];
#pragma unroll
            for (int i = 0; i < NCH; i++) {
                const int e0 = (lane + 64 * i) * 8;
                const u32x4 z = {0u, 0u, 0u, 0u};
                raw[i] = e0 < p.K ? ldg16(row + e0) : z;
            }
#pragma unroll
            for (int i = 0; i < NCH; i++) {
                if ((lane + 64 * i) * 8 < p.K) {
                    const half8v t = as_half8(raw[i]);
#pragma unroll
                    for (int j = 0; j < 8; j++) s += (float)t[j];
                }
            }
            s = wave_sum(s);
            const float mu = s / (float)p.K;
#pragma unroll
            for (int i = 0; i < NCH; i++) {
                if ((lane + 64 * i) * 8 < p.K) {
                    const half8v t = as_half8(raw[i]);
#pragma unroll
                    for (int j = 0; j < 8; j++) { const float d = (float)t[j] - mu; s2 = fmaf(d, d, s2); }
                }
            }
            s2 = wave_sum(s2);
            if (lane == 0) { stats[m][0] = mu; stats[m][1] = 1.0f / sqrtf(s2 / (float)p.K + p.ln_eps); }
        } else {
            for (int e0 = lane * 8; e0 < p.K; e0 += 512) {
                const half8v t = as_half8(ldg16(row + e0));
#pragma unroll
                for (int j = 0; j < 8; j++) s += (float)t[j];
            }
            s = wave_sum(s);
            const float mu = s / (float)p.K;
            for (int e0 = lane * 8; e0 < p.K; e0 += 512) {
                const half8v t = as_half8(ldg16(row + e0));
#pragma unroll
                for (int j = 0; j < 8; j++) { const float d = (float)t[j] - mu; s2 = fmaf(d, d, s2); }
            }
            s2 = wave_sum(s2);
            if (lane == 0) { stats[m][0] = mu; stats[m][1] = 1.0f / sqrtf(s2 / (float)p.K + p.ln_eps); }
        }
    }
}

// Eight activations of row statistics (mu, r) at column k0 of A, normalised and rounded as layernorm_vec_kernel does.
__device__ __forceinline__ u32x4 ln_apply8(const GemmArgs &p, u32x4 raw, float mu, float r, int k0) {
    const half8v x = as_half8(raw);
    half8v gv, bv, o;
    if (p.ln_gamma) gv = as_half8(ldg16(p.ln_gamma + k0));
    if (p.ln_beta) bv = as_half8(ldg16(p.ln_beta + k0));
#pragma unroll
    for (int j = 0; j < 8; j++)
        o[j] = ln_norm1((float)x[j], mu, r, p.ln_gamma != nullptr, p.ln_gamma ? (float)gv[j] : 0.0f, p.ln_beta != nullptr, p.ln_beta ? (float)bv[j] : 0.0f);
    return __builtin_bit_cast(u32x4, o);
}

// stage_args for the decode-sized kernels of [F][K] weights
__device__ __forceinline__ void stage_skinny(const GemmArgs &p) {
    asm volatile("" ::"s"(p.A), "s"(p.B), "s"(p.ldA), "s"(p.ldB), "s"(p.M), "s"(p.N), "s"(p.K), "s"(p.bias_mode), "s"(p.epi), "s"(p.Y), "s"(p.ldY), "s"(p.bias),
                 "s"(p.residual), "s"(p.out_f32), "s"(p.ln_gamma), "s"(p.ln_beta), "s"(p.ln_eps), "s"(p.ln_on), "s"(p.div_k8));
}

constexpr int SKN_COLS = 128;      // columns per workgroup
constexpr int SKN_KMAX = 256;      // deepest k-slice: 16 loads of 16 bytes per thread, all in flight at once
constexpr int SKN_LOADS = SKN_KMAX / 32;

template <int MT>
__global__ __launch_bounds__(256) void skinny_kn_kernel(GemmArgs p, float *part, int kper) {
    __shared__ __align__(16) half_t xs[MT][SKN_KMAX];
    __shared__ float red[4][MT][SKN_COLS];
    __shared__ float lnst[MT][2];
    const int tid = threadIdx.x, lane = tid & 63, wave = tid >> 6;
    const int cx = tid & 15, ky = tid >> 4;            // ky = 0..15: k-pairs 2 ky, 2 ky + 1 (+ 32 i)
    const int n = blockIdx.x * SKN_COLS + cx * 8;
    const int split = blockIdx.y;
    const int k0 = split * kper, klen = min(p.K - k0, kper);     // kper % 32 == 0, K % 8 == 0
    // weights first: they are what the memory system has to deliver
    u32x4 w[SKN_LOADS][2];
    const bool ncol = n < p.N;                          // NB % 8 == 0: a thread's 8 columns are in the row or all past N
    const half_t *bp = p.B + (long)k0 * p.ldB + n;
#pragma unroll
    for (int i = 0; i < SKN_LOADS; i++) {
        const int k = 32 * i + 2 * ky;
        const u32x4 z = {0u, 0u, 0u, 0u};
        if (32 * i < kper) {
            w[i][0] = (ncol && k < klen) ? ldg16(bp + (long)k * p.ldB) : z;
            w[i][1] = (ncol && k + 1 < klen) ? ldg16(bp + (long)(k + 1) * p.ldB) : z;
        }
    }
    if (p.ln_on) {                                      // uniform
        ln_row_stats<MT>(p, lnst, tid);
        __syncthreads();
    }
    for (int c = tid; c < MT * (kper >> 3); c += 256) {
        const int m = c / (kper >> 3), ch = c % (kper >> 3);
        u32x4 v = {0u, 0u, 0u, 0u};
        if (m < p.M && ch * 8 < klen) {
            v = ldg16(p.A + (long)m * p.ldA + k0 + ch * 8);
            if (p.ln_on) v = ln_apply8(p, v, lnst[m][0], lnst[m][1], k0 + ch * 8);
        }
        *reinterpret_cast<u32x4 *>(&xs[m][ch * 8]) = v;
    }
    __syncthreads();
    float acc[MT][8];
#pragma unroll
    for (int m = 0; m < MT; m++)
#pragma unroll
        for (int e = 0; e < 8; e++) acc[m][e] = 0.0f;
#pragma unroll
    for (int i = 0; i < SKN_LOADS; i++) {
        if (32 * i < kper) {
            const int k = 32 * i + 2 * ky;
            // (w[k][n+e], w[k+1][n+e]) pairs
            uint32_t pr[8];
#pragma unroll
            for (int q = 0; q < 4; q++) { pr[2 * q] = pack_lo(w[i][0][q], w[i][1][q]); pr[2 * q + 1] = pack_hi(w[i][0][q], w[i][1][q]); }
#pragma unroll
            for (int m = 0; m < MT; m++) {
                const half2v x = *reinterpret_cast<const half2v *>(&xs[m][k]);
#pragma unroll
                for (int e = 0; e < 8; e++) acc[m][e] = __builtin_amdgcn_fdot2(__builtin_bit_cast(half2v, pr[e]), x, acc[m][e], false);
            }
        }
    }
    // a wave holds 4 thread rows of the same 16 column groups: fold them, then the 4 waves through LDS
#pragma unroll
    for (int m = 0; m < MT; m++)
#pragma unroll
        for (int e = 0; e < 8; e++) {
            float v = acc[m][e];
            float x0 = v, y0 = v;
            swap_rows16(x0, y0); v = x0 + y0;            // v[lane] + v[lane ^ 16]
            x0 = v; y0 = v;
            swap_rows32(x0, y0); v = x0 + y0;            // ... + the same of lane ^ 32
            if (lane < 16) red[wave][m][cx * 8 + e] = v;
        }
    __syncthreads();
    for (int c = tid; c < MT * SKN_COLS; c += 256) {
        const int m = c / SKN_COLS, col = c % SKN_COLS;
        const int nn = blockIdx.x * SKN_COLS + col;
        if (m < p.M && nn < p.N) part[((long)split * p.M + m) * p.N + nn] = (red[0][m][col] + red[1][m][col]) + (red[2][m][col] + red[3][m][col]);
    }
}

// out[m][n] = epi(round(sum_s part[s][m][n] + bias)) (+ residual).  A thread's plane loads are
// issued eight at a time, so the sum costs a few memory round trips, not one per plane.
__global__ void skinny_epilogue_kernel(GemmArgs p, const float *part, int nsplit) {
    // (asked for at once, as stage_skinny does; 24 shapes of one to eight rows, both launches: 0.5 % faster.  The launch before it lost as much by it.)
    asm volatile("" ::"s"(p.M), "s"(p.N), "s"(p.bias_mode), "s"(p.epi), "s"(p.Y), "s"(p.ldY), "s"(p.bias), "s"(p.residual), "s"(p.out_f32), "s"(part), "s"(nsplit));
    long idx = (long)blockIdx.x * blockDim.x + threadIdx.x;
    long total = (long)p.M * p.N;
    if (idx >= total) return;
    int n = (int)(idx % p.N), m = (int)(idx / p.N);
    float v = p.bias_mode == MI_BIAS_COL ? (float)p.bias[n] : p.bias_mode == MI_BIAS_ROW ? (float)p.bias[m] : 0.0f;
    int s = 0;
    for (; s + 8 <= nsplit; s += 8) {
        float t[8];
#pragma unroll
        for (int j = 0; j < 8; j++) t[j] = part[(long)(s + j) * total + idx];
        v += ((t[0] + t[1]) + (t[2] + t[3])) + ((t[4] + t[5]) + (t[6] + t[7]));
    }
    for (; s < nsplit; s++) v += part[(long)s * total + idx];
    long off = (long)m * p.ldY + n;
    if (p.out_f32) reinterpret_cast<float *>(p.Y)[off] = apply_epi(v, p.epi);
    else {
        half_t o = (half_t)apply_epi((float)(half_t)v, p.epi);
        if (p.residual) o = (half_t)((float)o + (float)p.residual[off]);
        reinterpret_cast<half_t *>(p.Y)[off] = o;
    }
}

// [F][K] weights (K-contiguous): one wave per output column, lanes stride K in 16-byte chunks,
// wave reduction, and the epilogue in the same launch: no workspace, no second kernel.  The
// activations are staged in LDS once per workgroup (dynamic: MT rows of K halves).
//
// A decode-sized call moves a few MB, so its duration is a chain of trips to memory, not bandwidth.  Everything whose
// address does not depend on loaded data is therefore requested at the top, before anything is waited for: the wave's
// weight row (FK_PF chunks of 16 bytes per lane: K <= 6144 whole), its bias and residual elements, the thread's
// share of the activations and of gamma / beta.  The statistics of the layer-norm prologue, the staging and the dot
// products then run on data that arrives together: one trip instead of three or four in a row.
// FK_PF = 3 (K <= 1536) or 12: the registers of the up-front requests decide how many waves a SIMD holds, and a
// wide output (1280 -> 5120 is five waves per SIMD, a vocabulary projection many more) needs them all resident.
template <int MT, int FK_PF>
__global__ __launch_bounds__(256) void skinny_fk_kernel(GemmArgs p) {
    // activation chunks per thread requested up front: the whole MT x K panel up to four per thread
    constexpr int FK_XPF = (MT * FK_PF * 64 + 255) / 256 < 4 ? (MT * FK_PF * 64 + 255) / 256 : 4;
    extern __shared__ __align__(16) char smem[];
    stage_skinny(p);
    half_t *xs = reinterpret_cast<half_t *>(smem);       // [MT][K]
    const int tid = threadIdx.x, lane = tid & 63, wave = tid >> 6;
    __shared__ float lnst[MT][2];
    const int kch = p.K >> 3;
    const u32x4 z = {0u, 0u, 0u, 0u};
    const int n = blockIdx.x * 4 + wave;
    const bool live = n < p.N;                            // uniform over the wave
    const half_t *bp = p.B + (long)(live ? n : 0) * p.ldB;
    u32x4 w[FK_PF];
#pragma unroll
    for (int i = 0; i < FK_PF; i++) w[i] = live && lane * 8 + 512 * i < p.K ? ldg16(bp + lane * 8 + 512 * i) : z;
    float bv = 0.0f, rv = 0.0f;
    if (live && lane < p.M) {
        if (p.bias_mode == MI_BIAS_COL) bv = (float)p.bias[n];
        else if (p.bias_mode == MI_BIAS_ROW) bv = (float)p.bias[lane];
        if (p.residual && !p.out_f32) rv = (float)p.residual[(long)lane * p.ldY + n];
    }
    u32x4 xr[FK_XPF], gr[FK_XPF], br[FK_XPF];
#pragma unroll
    for (int i = 0; i < FK_XPF; i++) {
        unsigned ch;
        const int c = tid + 256 * i, m = (int)divide(c, kch, p.div_k8, ch);
        xr[i] = gr[i] = br[i] = z;
        if (c < MT * kch && m < p.M) {
            xr[i] = ldg16(p.A + (long)m * p.ldA + ch * 8);
            if (p.ln_on && p.ln_gamma) gr[i] = ldg16(p.ln_gamma + ch * 8);
            if (p.ln_on && p.ln_beta) br[i] = ldg16(p.ln_beta + ch * 8);
        }
    }
    if (p.ln_on) {                                      // uniform
        ln_row_stats<MT, (FK_PF < 8 ? FK_PF : 8)>(p, lnst, tid);
        __syncthreads();
    }
#pragma unroll
    for (int i = 0; i < FK_XPF; i++) {
        unsigned ch;
        const int c = tid + 256 * i, m = (int)divide(c, kch, p.div_k8, ch);
        if (c < MT * kch) {
            u32x4 v = xr[i];
            if (p.ln_on && m < p.M) {
                const half8v x = as_half8(v), gv = as_half8(gr[i]), bb = as_half8(br[i]);
                half8v o;
#pragma unroll
                for (int j = 0; j < 8; j++)
                    o[j] = ln_norm1((float)x[j], lnst[m][0], lnst[m][1], p.ln_gamma != nullptr, (float)gv[j], p.ln_beta != nullptr, (float)bb[j]);
                v = __builtin_bit_cast(u32x4, o);
            }
            *reinterpret_cast<u32x4 *>(xs + (long)m * p.K + ch * 8) = v;
        }
    }
    for (int c = tid + 256 * FK_XPF; c < MT * kch; c += 256) {
        unsigned ch;
        const int m = (int)divide(c, kch, p.div_k8, ch);
        u32x4 v = z;
        if (m < p.M) {
            v = ldg16(p.A + (long)m * p.ldA + ch * 8);
            if (p.ln_on) v = ln_apply8(p, v, lnst[m][0], lnst[m][1], ch * 8);
        }
        *reinterpret_cast<u32x4 *>(xs + (long)m * p.K + ch * 8) = v;
    }
    __syncthreads();
    if (!live) return;
    // A wave walks columns n, n + 4 gridDim.x, ...: one for the widths of a decoder layer (the launcher gives every
    // column its wave), several for a vocabulary-sized output, where the staged activations and their norm are then
    // paid once per workgroup instead of once per four columns and the next column's row is requested under the
    // current one's dot products.
    const int stride = (int)gridDim.x * 4;
    for (int nc = n; nc < p.N; nc += stride) {
        const int nn = nc + stride;
        const bool more = nn < p.N;                       // uniform over the wave
        const half_t *bn = p.B + (long)(more ? nn : nc) * p.ldB;
        u32x4 wn[FK_PF];
        float bvn = 0.0f, rvn = 0.0f;
        if (more) {
#pragma unroll
            for (int i = 0; i < FK_PF; i++) wn[i] = lane * 8 + 512 * i < p.K ? ldg16(bn + lane * 8 + 512 * i) : z;
            if (lane < p.M) {
                if (p.bias_mode == MI_BIAS_COL) bvn = (float)p.bias[nn];
                else if (p.bias_mode == MI_BIAS_ROW) bvn = (float)p.bias[lane];
                if (p.residual && !p.out_f32) rvn = (float)p.residual[(long)lane * p.ldY + nn];
            }
        }
        float acc[MT];
#pragma unroll
        for (int m = 0; m < MT; m++) acc[m] = 0.0f;
        auto dot = [&](const u32x4 &wv, int k) {
#pragma unroll
            for (int m = 0; m < MT; m++) {
                const u32x4 x = *reinterpret_cast<const u32x4 *>(xs + (long)m * p.K + k);
#pragma unroll
                for (int q = 0; q < 4; q++) {
                    const uint32_t wq = wv[q], xq = x[q];     // bit_cast wants an addressable scalar, not a vector element
                    acc[m] = __builtin_amdgcn_fdot2(__builtin_bit_cast(half2v, wq), __builtin_bit_cast(half2v, xq), acc[m], false);
                }
            }
        };
#pragma unroll
        for (int i = 0; i < FK_PF; i++)
            if (lane * 8 + 512 * i < p.K) dot(w[i], lane * 8 + 512 * i);
        const half_t *bc = p.B + (long)nc * p.ldB;
        for (int kb = lane * 8 + 512 * FK_PF; kb < p.K; kb += 4 * 512) {
            u32x4 t[4];
#pragma unroll
            for (int i = 0; i < 4; i++) t[i] = kb + 512 * i < p.K ? ldg16(bc + kb + 512 * i) : z;
#pragma unroll
            for (int i = 0; i < 4; i++)
                if (kb + 512 * i < p.K) dot(t[i], kb + 512 * i);
        }
        float mine = 0.0f;                                    // lane m keeps row m's sum
#pragma unroll
        for (int m = 0; m < MT; m++) {
            float sres = acc[m];
            sres = wave_sum(sres);
            if (lane == m) mine = sres;
        }
        if (lane < p.M) {
            const float v = mine + bv;
            const long off = (long)lane * p.ldY + nc;
            if (p.out_f32) reinterpret_cast<float *>(p.Y)[off] = apply_epi(v, p.epi);
            else {
                half_t o = (half_t)apply_epi((float)(half_t)v, p.epi);
                if (p.residual) o = (half_t)((float)o + rv);
                reinterpret_cast<half_t *>(p.Y)[off] = o;
            }
        }
        if (more) {
#pragma unroll
            for (int i = 0; i < FK_PF; i++) w[i] = wn[i];
            bv = bvn; rv = rvn;
        }
    }
}

// Five to eight rows: on the matrix cores.  A workgroup owns sixteen output columns (`cols`; eight where that gives more CUs work), its
// eight waves an eighth of K each: the weight rows by 32 k are one operand of v_mfma_f32_16x16x32_f16, the activation rows the
// other (zeros past either), both straight from memory in the layout the instruction wants -- a lane's sixteen bytes -- and all of a wave's share asked for at its first
// lines (PF steps at a time).  The eight partial sums meet in LDS, in pairs.  With a norm in front a wave finds one row's statistics,
// in layernorm_vec_kernel's order, and the fragments are normalised and rounded on their way into the product.
// What bounds it is the trip to memory.  The kernel above staged M x K activations in every workgroup of four columns and read them back
// once a column: 80 KB of LDS traffic a wave at 8 x 5120.
template <int PF, bool LN>
__global__ __launch_bounds__(512) void few_rows_kernel(GemmArgs p, int cols) {
    constexpr int NW = 8;
    __shared__ float4v red[NW][64];
    __shared__ float lnst[8][2];
    stage_skinny(p);
    const int tid = threadIdx.x, lane = tid & 63, wave = __builtin_amdgcn_readfirstlane(tid >> 6);
    const int row = lane & 15, kq = lane >> 4, n0 = blockIdx.x * cols;
    const int steps = (p.K + 31) >> 5, per = (steps + NW - 1) / NW, s0 = wave * per, s1 = min(steps, s0 + per);
    const half_t *const wrow = p.B + (long)min(n0 + row, p.N - 1) * p.ldB, *const xrow = p.A + (long)min(row, p.M - 1) * p.ldA;
    u32x4 w[PF], x[PF], g[LN ? PF : 1], b[LN ? PF : 1];
    auto fetch = [&](int base) {
#pragma unroll
        for (int i = 0; i < PF; i++) {
            const u32x4 z = {0u, 0u, 0u, 0u};
            const int k = (base + i) * 32 + kq * 8;
            const bool on = base + i < s1 && k < p.K;
            w[i] = on && row < cols ? ldg16(wrow + k) : z;
            x[i] = on && row < p.M ? ldg16(xrow + k) : z;
            if constexpr (LN) {
                // (columns that are not there have gamma zero, whatever the row's mean: as a half it may be an infinity)
                const u32x4 ones = {0x3c003c00u, 0x3c003c00u, 0x3c003c00u, 0x3c003c00u};
                g[i] = !on ? z : p.ln_gamma ? ldg16(p.ln_gamma + k) : ones;
                b[i] = on && p.ln_beta ? ldg16(p.ln_beta + k) : z;
            }
        }
    };
    fetch(s0);
    // what the store needs, by the wave that stores: lane (row, kq) holds columns n0 + 4 kq .. +3 of row `row`
    const int n = n0 + 4 * kq;
    const bool stores = wave == 0 && row < p.M && 4 * kq < cols;
    float bv[4] = {0.0f, 0.0f, 0.0f, 0.0f}, rv[4] = {0.0f, 0.0f, 0.0f, 0.0f};
    if (stores) {
#pragma unroll
        for (int e = 0; e < 4; e++) {
            if (n + e < p.N) {
                if (p.bias_mode == MI_BIAS_COL) bv[e] = (float)p.bias[n + e];
                else if (p.bias_mode == MI_BIAS_ROW) bv[e] = (float)p.bias[row];
                if (p.residual && !p.out_f32) rv[e] = (float)p.residual[(long)row * p.ldY + n + e];
            }
        }
    }
    float mu = 0.0f, rs = 0.0f;
    if constexpr (LN) {
        ln_row_stats<8, 8, NW>(p, lnst, tid);
        __syncthreads();
        mu = lnst[min(row, p.M - 1)][0];
        rs = lnst[min(row, p.M - 1)][1];
    }
    // five chains, step i of the share in chain i % 5 whatever PF is: short ones keep the error at that of the dot products below five rows
    constexpr int NA = 5;
    static_assert(PF % NA == 0, "one order of the sum, with a norm in front and without");
    float4v acc[NA];
#pragma unroll
    for (int i = 0; i < NA; i++) acc[i] = float4v{0.0f, 0.0f, 0.0f, 0.0f};
    for (int base = s0;;) {
#pragma unroll
        for (int i = 0; i < PF; i++) {
            half8v xv = as_half8(x[i]);
            if constexpr (LN) {
                const half8v gv = as_half8(g[i]), be = as_half8(b[i]);
#pragma unroll
                for (int j = 0; j < 8; j++) xv[j] = ln_norm1((float)xv[j], mu, rs, true, (float)gv[j], p.ln_beta != nullptr, (float)be[j]);
            }
            acc[i % NA] = __builtin_amdgcn_mfma_f32_16x16x32_f16(as_half8(w[i]), xv, acc[i % NA], 0, 0, 0);      // (steps past the share multiply zeros)
        }
        if ((base += PF) >= s1) break;
        fetch(base);
    }
#pragma unroll
    for (int d = 1; d < NA; d *= 2)
#pragma unroll
        for (int i = 0; i + d < NA; i += 2 * d) acc[i] += acc[i + d];
    red[wave][lane] = acc[0];
    __syncthreads();
    if (!stores) return;
    float4v sum[NW];
#pragma unroll
    for (int q = 0; q < NW; q++) sum[q] = red[q][lane];
#pragma unroll
    for (int d = 1; d < NW; d *= 2)
#pragma unroll
        for (int q = 0; q < NW; q += 2 * d) sum[q] += sum[q + d];
    const float4v v = sum[0];
#pragma unroll
    for (int e = 0; e < 4; e++) {
        if (n + e < p.N) {
            const float t = v[e] + bv[e];
            const long off = (long)row * p.ldY + n + e;
            if (p.out_f32) reinterpret_cast<float *>(p.Y)[off] = apply_epi(t, p.epi);
            else {
                half_t o = (half_t)apply_epi((float)(half_t)t, p.epi);
                if (p.residual) o = (half_t)((float)o + rv[e]);
                reinterpret_cast<half_t *>(p.Y)[off] = o;
            }
        }
    }
}

// The same product with the activations in registers instead of LDS, for the few rows of a decode step: a lane's
// weight chunks sit at k = 8 lane + 512 i, so it needs exactly those chunks of every activation row and asks for
// them itself (the rows come from the L2: every wave of the launch reads the same few KB).  No staging, no barrier:
// a wave is a chain of one trip to memory, the norm statistics (its own copy, same summation order as
// ln_row_stats, so the same bits), the dot products, one wave reduction and a store.  R output columns per wave,
// all their weight rows requested up front.  (MT + R + 2) * PF chunks of registers: built for one and two rows of
// K <= 1536 (78 to 119 registers, four to six waves per SIMD); four rows, or K = 5120, would leave a SIMD one or
// two waves and stay with the staged kernel.
template <int MT, int PF, int R>
__global__ __launch_bounds__(256) void skinny_fk_reg_kernel(GemmArgs p) {
    stage_skinny(p);
    const int lane = threadIdx.x & 63, wave = threadIdx.x >> 6;
    const u32x4 z = {0u, 0u, 0u, 0u};
    const int n0 = (blockIdx.x * 4 + wave) * R;
    if (n0 >= p.N) return;                                // uniform over the wave; no barrier below
    u32x4 w[R][PF];
#pragma unroll
    for (int r = 0; r < R; r++) {
        const half_t *bp = p.B + (long)min(n0 + r, p.N - 1) * p.ldB;
#pragma unroll
        for (int i = 0; i < PF; i++) w[r][i] = lane * 8 + 512 * i < p.K ? ldg16(bp + lane * 8 + 512 * i) : z;
    }
    u32x4 x[MT][PF], gr[PF], br[PF];
#pragma unroll
    for (int i = 0; i < PF; i++) {
        const int k = lane * 8 + 512 * i;
        gr[i] = br[i] = z;
#pragma unroll
        for (int m = 0; m < MT; m++) x[m][i] = m < p.M && k < p.K ? ldg16(p.A + (long)m * p.ldA + k) : z;
        if (p.ln_on && k < p.K) {
            if (p.ln_gamma) gr[i] = ldg16(p.ln_gamma + k);
            if (p.ln_beta) br[i] = ldg16(p.ln_beta + k);
        }
    }
    float bv[R], rv[R];
#pragma unroll
    for (int r = 0; r < R; r++) {
        bv[r] = rv[r] = 0.0f;
        if (lane < p.M && n0 + r < p.N) {
            if (p.bias_mode == MI_BIAS_COL) bv[r] = (float)p.bias[n0 + r];
            else if (p.bias_mode == MI_BIAS_ROW) bv[r] = (float)p.bias[lane];
            if (p.residual && !p.out_f32) rv[r] = (float)p.residual[(long)lane * p.ldY + n0 + r];
        }
    }
    if (p.ln_on) {                                        // uniform
#pragma unroll
        for (int m = 0; m < MT; m++) {
            float s1 = 0.0f, s2 = 0.0f;
#pragma unroll
            for (int i = 0; i < PF; i++) {
                if (lane * 8 + 512 * i < p.K) {
                    const half8v t = as_half8(x[m][i]);
#pragma unroll
                    for (int j = 0; j < 8; j++) s1 += (float)t[j];
                }
            }
            s1 = wave_sum(s1);
            const float mu = s1 / (float)p.K;
#pragma unroll
            for (int i = 0; i < PF; i++) {
                if (lane * 8 + 512 * i < p.K) {
                    const half8v t = as_half8(x[m][i]);
#pragma unroll
                    for (int j = 0; j < 8; j++) { const float d = (float)t[j] - mu; s2 = fmaf(d, d, s2); }
                }
            }
            s2 = wave_sum(s2);
            const float rs = 1.0f / sqrtf(s2 / (float)p.K + p.ln_eps);
#pragma unroll
            for (int i = 0; i < PF; i++) {
                const half8v t = as_half8(x[m][i]), gv = as_half8(gr[i]), bb = as_half8(br[i]);
                half8v o;
#pragma unroll
                for (int j = 0; j < 8; j++) o[j] = ln_norm1((float)t[j], mu, rs, p.ln_gamma != nullptr, (float)gv[j], p.ln_beta != nullptr, (float)bb[j]);
                x[m][i] = lane * 8 + 512 * i < p.K ? __builtin_bit_cast(u32x4, o) : z;
            }
        }
    }
    float acc[R][MT];
#pragma unroll
    for (int r = 0; r < R; r++)
#pragma unroll
        for (int m = 0; m < MT; m++) acc[r][m] = 0.0f;
#pragma unroll
    for (int i = 0; i < PF; i++)
#pragma unroll
        for (int r = 0; r < R; r++)
#pragma unroll
            for (int m = 0; m < MT; m++)
#pragma unroll
                for (int q = 0; q < 4; q++) {
                    const uint32_t wq = w[r][i][q], xq = x[m][i][q];
                    acc[r][m] = __builtin_amdgcn_fdot2(__builtin_bit_cast(half2v, wq), __builtin_bit_cast(half2v, xq), acc[r][m], false);
                }
#pragma unroll
    for (int r = 0; r < R; r++) {
        float mine = 0.0f;                                // lane m keeps row m's sum
#pragma unroll
        for (int m = 0; m < MT; m++) {
            const float sres = wave_sum(acc[r][m]);
            if (lane == m) mine = sres;
        }
        if (lane < p.M && n0 + r < p.N) {
            const float v = mine + bv[r];
            const long off = (long)lane * p.ldY + n0 + r;
            if (p.out_f32) reinterpret_cast<float *>(p.Y)[off] = apply_epi(v, p.epi);
            else {
                half_t o = (half_t)apply_epi((float)(half_t)v, p.epi);
                if (p.residual) o = (half_t)((float)o + rv[r]);
                reinterpret_cast<half_t *>(p.Y)[off] = o;
            }
        }
    }
}

// k-slice depth for the [K][F] skinny kernel: enough workgroups to put ~2 on every CU, slices a
// multiple of 32 within [64, SKN_KMAX].
int skinny_kper(int64_t K, int64_t F) {
    const int64_t colblocks = ceil_div(F, SKN_COLS);
    const int64_t want = ceil_div(2 * (int64_t)mi_num_cus(), colblocks);
    int64_t kper = (int64_t)round_up((size_t)ceil_div(K, want), 32);
    if (kper < 64) kper = 64;
    if (kper > SKN_KMAX) kper = SKN_KMAX;
    return (int)kper;
}

// few_rows_kernel from five rows on (us at 4 and 8 rows, staged kernel | matrix cores; 1280 -> 5120 6.8 | 7.15 and 8.6 | 7.4; 4096 -> 1024
// 6.4 | 7.1 and 10.3 | 7.9; 5120 -> 1280 8.9 | 8.2 and 20.4 | 9.0; 1280 -> 51866 35.8 | 35.0 and 48 | 38; 1536 -> 384 3.8 | 4.4 and 4.9 | 4.65).
constexpr int FEW_ROWS_MIN = 5;

}  // namespace

int mi_skinny_splits(int64_t K, int64_t F) { return (int)ceil_div(K, skinny_kper(K, F)); }

int mi_skinny_launch(const GemmArgs &a, bool b_kn, void *ws, size_t ws_bytes, hipStream_t st) {
    if (b_kn) {
        const int kper = skinny_kper(a.K, a.N), nsplit = (int)ceil_div(a.K, kper);
        size_t need = (size_t)nsplit * a.M * a.N * sizeof(float);
        if (!ws || ws_bytes < need || !aligned_to(ws, 256)) return MI_DECLINE_WORKSPACE;
        float *part = reinterpret_cast<float *>(ws);
        dim3 grid((unsigned)ceil_div(a.N, SKN_COLS), (unsigned)nsplit);
        if (a.M <= 1)      hipLaunchKernelGGL(skinny_kn_kernel<1>, grid, dim3(256), 0, st, a, part, kper);
        else if (a.M <= 2) hipLaunchKernelGGL(skinny_kn_kernel<2>, grid, dim3(256), 0, st, a, part, kper);
        else if (a.M <= 4) hipLaunchKernelGGL(skinny_kn_kernel<4>, grid, dim3(256), 0, st, a, part, kper);
        else if (a.M <= 8) hipLaunchKernelGGL(skinny_kn_kernel<8>, grid, dim3(256), 0, st, a, part, kper);
        else return MI_DECLINE_EXTENT;
        long total = (long)a.M * a.N;
        hipLaunchKernelGGL(skinny_epilogue_kernel, dim3((unsigned)ceil_div(total, 256)), dim3(256), 0, st, a, part, nsplit);
    } else {
        const int mt = a.M <= 1 ? 1 : a.M <= 2 ? 2 : 4;
        const size_t lds = (size_t)mt * a.K * sizeof(half_t);
        if (a.M > 8 || lds > SKINNY_FK_LDS_MAX) return MI_DECLINE_EXTENT;
        if (a.M >= FEW_ROWS_MIN) {
            const int cols = ceil_div(a.N, 16) * 2 <= mi_num_cus() ? 8 : 16, per = (int)ceil_div(ceil_div(a.K, 32), 8);
            const dim3 grid((unsigned)ceil_div(a.N, cols));
            if (a.ln_on) {
                if (per <= 5) hipLaunchKernelGGL((few_rows_kernel<5, true>), grid, dim3(512), 0, st, a, cols);
                else          hipLaunchKernelGGL((few_rows_kernel<10, true>), grid, dim3(512), 0, st, a, cols);
            } else {
                if (per <= 5)       hipLaunchKernelGGL((few_rows_kernel<5, false>), grid, dim3(512), 0, st, a, cols);
                else if (per <= 10) hipLaunchKernelGGL((few_rows_kernel<10, false>), grid, dim3(512), 0, st, a, cols);
                else                hipLaunchKernelGGL((few_rows_kernel<20, false>), grid, dim3(512), 0, st, a, cols);
            }
            return hipGetLastError() == hipSuccess ? MI_OK : MI_ERROR_LAUNCH;
        }
        // rows per wave: as many as still leave every CU a workgroup, at most eight (a workgroup stages
        // all M activation rows once, whatever the number of weight rows it then streams)
        // One weight row per wave.  More rows per wave would amortise the staging of the activations, but the
        // rows of a wave run one after the other, each a chain of dependent memory trips: measured slower at
        // every batch size (1280 -> 5120, batch 8: 9.1 us with one row, 13.7 us with four).
        // One or two rows without a norm in front: activations in registers, no staging (hot in a replayed graph at
        // batch 1: 2.88 / 3.13 / 3.34 us for 1280 -> 1280 / 3840 / 5120 against 3.01 / 3.33 / 3.57 us staged).  With
        // the layer-norm prologue every wave would normalise its own copy of the row -- 4.5 / 6.1 / 6.9 us against
        // 3.9 / 4.3 / 4.7 us -- so that stays staged, and so does a very wide output (51866 columns: 24.5 against 23.0 us).
        int R = 1;
        if (!a.ln_on && a.N <= 8192 && a.K <= 1536 && mt <= 2) {
            dim3 rg((unsigned)ceil_div(a.N, 4 * R));
            if (R == 2) {
                if (mt == 1)      hipLaunchKernelGGL((skinny_fk_reg_kernel<1, 3, 2>), rg, dim3(256), 0, st, a);
                else              hipLaunchKernelGGL((skinny_fk_reg_kernel<2, 3, 2>), rg, dim3(256), 0, st, a);
            } else {
                if (mt == 1)      hipLaunchKernelGGL((skinny_fk_reg_kernel<1, 3, 1>), rg, dim3(256), 0, st, a);
                else              hipLaunchKernelGGL((skinny_fk_reg_kernel<2, 3, 1>), rg, dim3(256), 0, st, a);
            }
            return hipGetLastError() == hipSuccess ? MI_OK : MI_ERROR_LAUNCH;
        }
        // every column its own wave up to eight workgroups per CU; beyond that (a vocabulary projection) a wave walks
        // several columns behind one staging of the activations
        const int64_t wgs = ceil_div(a.N, 4), cap = (int64_t)mi_num_cus() * 8;
        dim3 grid((unsigned)(wgs < cap ? wgs : cap));
        if (a.K <= 1536) {
            if (mt == 1)      hipLaunchKernelGGL((skinny_fk_kernel<1, 3>), grid, dim3(256), lds, st, a);
            else if (mt == 2) hipLaunchKernelGGL((skinny_fk_kernel<2, 3>), grid, dim3(256), lds, st, a);
            else              hipLaunchKernelGGL((skinny_fk_kernel<4, 3>), grid, dim3(256), lds, st, a);
        } else {
            if (mt == 1)      hipLaunchKernelGGL((skinny_fk_kernel<1, 12>), grid, dim3(256), lds, st, a);
            else if (mt == 2) hipLaunchKernelGGL((skinny_fk_kernel<2, 12>), grid, dim3(256), lds, st, a);
            else              hipLaunchKernelGGL((skinny_fk_kernel<4, 12>), grid, dim3(256), lds, st, a);
        }
    }
    return hipGetLastError() == hipSuccess ? MI_OK : MI_ERROR_LAUNCH;
}

int mi_skinny_init() {
    int bad = 0;
    bad |= raise_lds(skinny_fk_kernel<1, 3>, (int)SKINNY_FK_LDS_MAX);
    bad |= raise_lds(skinny_fk_kernel<2, 3>, (int)SKINNY_FK_LDS_MAX);
    bad |= raise_lds(skinny_fk_kernel<4, 3>, (int)SKINNY_FK_LDS_MAX);
    bad |= raise_lds(skinny_fk_kernel<1, 12>, (int)SKINNY_FK_LDS_MAX);
    bad |= raise_lds(skinny_fk_kernel<2, 12>, (int)SKINNY_FK_LDS_MAX);
    bad |= raise_lds(skinny_fk_kernel<4, 12>, (int)SKINNY_FK_LDS_MAX);
    return bad;
}
