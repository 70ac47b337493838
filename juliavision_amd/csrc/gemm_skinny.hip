// fp16 GEMM for gfx950, decode-sized: up to eight rows of activations against weights of either layout, with a layer norm of the
// rows in front or without.
#include "gemm_common.hpp"

namespace {

// Decode-sized M (<= 8): bandwidth- and latency-bound.  Every weight byte is read once with
// 16-byte loads, a thread's loads are all issued before the first is used, and the activations
// (a few KB) are staged in LDS.  Products go through v_dot2_f32_f16: fp16 pairs, fp32 sum.

// Layer-norm statistics of up to MT rows of A, one wave per row, in the summation order of
// layernorm_vec_kernel (a lane takes the 16-byte chunks lane, lane + 64, ...; butterfly over the wave):
// the fused result is bit-identical to running that kernel first.  stats[m] = (mean, rstd).
// In two halves, so that a caller can ask for more in between (LnRow).  Rows up to NCH * 512 halves stay in registers between the
// passes; a longer one is read twice.  The two ways share no line but the last: where both led through one body, held and walked
// rows were live over the choice and took skinny_kn_kernel<8> from 156 registers to 194, a third of its waves (8 rows of 8944 -> 7608
// 41.6 -> 48.0 us, behind a norm 96 -> 129; 5 of 1464 -> 4248 11.1 -> 13.4).
__device__ __forceinline__ void ln_stats_done(const GemmArgs &p, float (*stats)[2], int m, int lane, float mu, float s2) {
    s2 = wave_sum(s2);
    if (lane == 0) { stats[m][0] = mu; stats[m][1] = 1.0f / sqrtf(s2 / (float)p.K + p.ln_eps); }
}
__device__ __forceinline__ void ln_stats_walked(const GemmArgs &p, float (*stats)[2], int m, int lane) {
    float s = 0.0f, s2 = 0.0f;
    const half_t *row = p.A + (long)m * p.ldA;
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
    ln_stats_done(p, stats, m, lane, mu, s2);
}
template <int NCH>
struct LnRow {
    u32x4 raw[NCH];
    __device__ __forceinline__ void load(const GemmArgs &p, int m, int lane) {
        const half_t *row = p.A + (long)m * p.ldA;
#pragma unroll
        for (int i = 0; i < NCH; i++) raw[i] = ldg16(row + min((lane + 64 * i) * 8, p.K - 8));
    }
    __device__ __forceinline__ void held(const GemmArgs &p, float (*stats)[2], int m, int lane) const {
        float s = 0.0f, s2 = 0.0f;
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
        ln_stats_done(p, stats, m, lane, mu, s2);
    }
    __device__ __forceinline__ void request(const GemmArgs &p, int m, int lane) { if (p.K <= NCH * 512) load(p, m, lane); }      // uniform
    __device__ __forceinline__ void finish(const GemmArgs &p, float (*stats)[2], int m, int lane) const {
        if (p.K <= NCH * 512) held(p, stats, m, lane);
        else ln_stats_walked(p, stats, m, lane);
    }
};
template <int MT, int NCH = 8, int NWAVES = 4>
__device__ __forceinline__ void ln_row_stats(const GemmArgs &p, float (*stats)[2], int tid) {
    const int lane = tid & 63, wave = tid >> 6;
    for (int m = wave; m < MT && m < p.M; m += NWAVES) {
        if (p.K <= NCH * 512) {
            LnRow<NCH> row;
            row.load(p, m, lane);
            row.held(p, stats, m, lane);
        } else ln_stats_walked(p, stats, m, lane);
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

// [K][F] weights that kn_on_tiles leaves here (K from 1280, of one or two rows from 768, and very wide outputs): a thread owns 8
// consecutive columns, 16 threads span 128 columns, the 16 thread rows of a workgroup take interleaved k-pairs.  K is split over
// workgroups so that the whole chip pulls on HBM; each split writes an fp32 partial plane and skinny_epilogue_kernel sums the
// planes (the reference's split-K planes + mm_epilogue_kernel!, matmul.jl:192-217).
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

// [F][K] weights (K-contiguous): one wave per R output columns, lanes stride K in 16-byte chunks,
// wave reduction, and the epilogue in the same launch: no workspace, no second kernel.
//
// A decode-sized call moves a few MB, so its duration is a chain of trips to memory, not bandwidth: everything whose
// address does not depend on loaded data is requested at the top, before anything is waited for.  For that no load may stand
// behind a condition -- where the registers of the two sides meet the compiler waits for the load, and with it, as loads come back
// in the order they were asked for, for every load before it (the bias, behind `if (lane < M)`, cost a trip of its own, the
// residual another, the activations a third: 1280 -> 1280 behind a norm 3.57 us, hot in a replayed graph).  So every address is made
// valid instead -- chunks past K re-read the row's last one, columns past N the last row, an operand that is not there the
// weights -- and what was read in vain is left out where it would be used.
// Bias and residual of the output of lane r * MT + m: row m of a wave's column r.
template <int MT, int R>
struct FkOut {
    half_t bias, residual;
    __device__ __forceinline__ void request(const GemmArgs &p, int n0, int lane) {
        const int m = min(lane % MT, p.M - 1), n = min(n0 + min(lane / MT, R - 1), p.N - 1);
        const half_t *b = p.bias_mode == MI_BIAS_NONE ? p.B : p.bias + (p.bias_mode == MI_BIAS_COL ? n : m);
        const half_t *r = p.residual && !p.out_f32 ? p.residual + (long)m * p.ldY + n : p.B;
        bias = *b;
        residual = *r;
    }
    __device__ __forceinline__ void store(const GemmArgs &p, float sum, int n0, int lane) const {
        const int m = lane % MT, n = n0 + lane / MT;
        if (lane >= MT * R || m >= p.M || n >= p.N) return;
        const float v = sum + (p.bias_mode == MI_BIAS_NONE ? 0.0f : (float)bias);
        const long off = (long)m * p.ldY + n;
        if (p.out_f32) reinterpret_cast<float *>(p.Y)[off] = apply_epi(v, p.epi);
        else {
            half_t o = (half_t)apply_epi((float)(half_t)v, p.epi);
            if (p.residual) o = (half_t)((float)o + (float)residual);
            reinterpret_cast<half_t *>(p.Y)[off] = o;
        }
    }
};
template <int R, int PF>
__device__ __forceinline__ void fk_request(const GemmArgs &p, u32x4 (&w)[R][PF], int n0, int lane) {
#pragma unroll
    for (int r = 0; r < R; r++) {
        const half_t *bp = p.B + (long)min(n0 + r, p.N - 1) * p.ldB;
#pragma unroll
        for (int i = 0; i < PF; i++) w[r][i] = ldg16(bp + min(lane * 8 + 512 * i, p.K - 8));
    }
}
__device__ __forceinline__ float fk_dot(u32x4 w, u32x4 x, float acc) {
#pragma unroll
    for (int q = 0; q < 4; q++) {
        const uint32_t wq = w[q], xq = x[q];              // bit_cast wants an addressable scalar, not a vector element
        acc = __builtin_amdgcn_fdot2(__builtin_bit_cast(half2v, wq), __builtin_bit_cast(half2v, xq), acc, false);
    }
    return acc;
}

// The activations staged in LDS once per workgroup (dynamic: MT rows of K halves), behind the layer norm of their rows (LN).
// PF: 512-column chunks of a row asked for at the top, all of K up to 6144.  R columns a wave: the norm, the staging and their two
// barriers are paid once a workgroup, so behind a norm a wave takes as many as leave one workgroup a CU (us, weights from memory, with 1
// and with R columns: 1280 -> 1280 3.9 and 3.5, -> 3840 5.2 and 4.2, -> 5120 5.6 and 4.7); without one the launch gains nothing by it.
template <int MT, int PF, int R, bool LN>
__global__ __launch_bounds__(256) void skinny_fk_kernel(GemmArgs p) {
    // activation chunks per thread requested up front: the whole MT x K panel, up to twelve per thread (four behind a norm: gamma and beta come with them)
    constexpr int XPF_MAX = LN ? 4 : 12, XPF = (MT * PF * 64 + 255) / 256 < XPF_MAX ? (MT * PF * 64 + 255) / 256 : XPF_MAX;
    extern __shared__ __align__(16) char smem[];
    stage_skinny(p);
    half_t *xs = reinterpret_cast<half_t *>(smem);       // [MT][K]
    const int tid = threadIdx.x, lane = tid & 63, wave = __builtin_amdgcn_readfirstlane(tid >> 6);
    __shared__ float lnst[MT][2];
    const int kch = p.K >> 3, staged = p.M * kch;         // (rows past M are not: their sums go nowhere)
    // what the norm and the staging wait for goes first
    LnRow<PF <= 10 ? PF : 8> lnrow;
    if constexpr (LN) lnrow.request(p, min(wave, p.M - 1), lane);      // (MT is at most the workgroup's four waves)
    u32x4 xr[XPF], gr[LN ? XPF : 1], br[LN ? XPF : 1];
#pragma unroll
    for (int i = 0; i < XPF; i++) {
        unsigned ch;
        const int c = tid + 256 * i, m = (int)divide(c, kch, p.div_k8, ch);
        xr[i] = ldg16(p.A + (long)min(m, p.M - 1) * p.ldA + ch * 8);
        if constexpr (LN) {
            gr[i] = ldg16((p.ln_gamma ? p.ln_gamma : p.A) + ch * 8);
            br[i] = ldg16((p.ln_beta ? p.ln_beta : p.A) + ch * 8);
        }
    }
    const int n = (blockIdx.x * 4 + wave) * R;
    u32x4 w[R][PF];
    FkOut<MT, R> out;
    fk_request(p, w, n, lane);
    out.request(p, n, lane);
    __builtin_amdgcn_sched_barrier(0);
    if constexpr (LN) {
        if (wave < p.M) lnrow.finish(p, lnst, wave, lane);
        __syncthreads();
    }
#pragma unroll
    for (int i = 0; i < XPF; i++) {
        unsigned ch;
        const int c = tid + 256 * i, m = (int)divide(c, kch, p.div_k8, ch);
        if (c < staged) {
            u32x4 v = xr[i];
            if constexpr (LN) {
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
    for (int c = tid + 256 * XPF; c < staged; c += 256) {
        unsigned ch;
        const int m = (int)divide(c, kch, p.div_k8, ch);
        u32x4 v = ldg16(p.A + (long)m * p.ldA + ch * 8);
        if constexpr (LN) v = ln_apply8(p, v, lnst[m][0], lnst[m][1], ch * 8);
        *reinterpret_cast<u32x4 *>(xs + (long)m * p.K + ch * 8) = v;
    }
    __syncthreads();
    // A wave walks its columns n .. n + R - 1, then those 4 R gridDim.x further on: once for the widths of a decoder layer
    // (the launcher gives every group its wave), several times for a vocabulary-sized output, where the staged activations
    // and their norm are then paid once per workgroup and the next rows are requested under the current ones' dot products.
    if (n >= p.N) return;                                 // uniform over the wave
    const int stride = (int)gridDim.x * 4 * R;
    for (int nc = n;; nc += stride) {
        u32x4 wn[R][PF];
        FkOut<MT, R> outn;
        const bool more = p.N - nc > stride;              // (past the end: the last row once more)
        const int nn = more ? nc + stride : p.N - 1;
        fk_request(p, wn, nn, lane);
        outn.request(p, nn, lane);
        float acc[R][MT];
#pragma unroll
        for (int r = 0; r < R; r++)
#pragma unroll
            for (int m = 0; m < MT; m++) acc[r][m] = 0.0f;
#pragma unroll
        for (int i = 0; i < PF; i++)
            if (lane * 8 + 512 * i < p.K) {
#pragma unroll
                for (int m = 0; m < MT; m++) {
                    const u32x4 x = *reinterpret_cast<const u32x4 *>(xs + (long)m * p.K + lane * 8 + 512 * i);
#pragma unroll
                    for (int r = 0; r < R; r++) acc[r][m] = fk_dot(w[r][i], x, acc[r][m]);
                }
            }
        if (p.K > 512 * PF)                               // uniform
#pragma unroll
            for (int r = 0; r < R; r++) {
                const half_t *bc = p.B + (long)min(nc + r, p.N - 1) * p.ldB;
                for (int kb = lane * 8 + 512 * PF; kb < p.K; kb += 4 * 512) {
                    u32x4 t[4];
#pragma unroll
                    for (int i = 0; i < 4; i++) t[i] = ldg16(bc + min(kb + 512 * i, p.K - 8));
#pragma unroll
                    for (int i = 0; i < 4; i++)
                        if (kb + 512 * i < p.K)
#pragma unroll
                            for (int m = 0; m < MT; m++) acc[r][m] = fk_dot(t[i], *reinterpret_cast<const u32x4 *>(xs + (long)m * p.K + kb + 512 * i), acc[r][m]);
                }
            }
        float mine = 0.0f;                                // lane r * MT + m keeps its sum
#pragma unroll
        for (int r = 0; r < R; r++)
#pragma unroll
            for (int m = 0; m < MT; m++) {
                const float sres = wave_sum(acc[r][m]);
                if (lane == r * MT + m) mine = sres;
            }
        out.store(p, mine, nc, lane);
        if (!more) break;
#pragma unroll
        for (int r = 0; r < R; r++)
#pragma unroll
            for (int i = 0; i < PF; i++) w[r][i] = wn[r][i];
        out = outn;
    }
}

// Five to eight rows: on the matrix cores.  A workgroup owns sixteen output columns (`cols`; eight where that gives more CUs work), its
// eight waves an eighth of K each: the weight rows by 32 k are one operand of v_mfma_f32_16x16x32_f16, the activation rows the
// other, both straight from memory in the layout the instruction wants -- a lane's sixteen bytes -- and all of a wave's share asked for at its first
// lines (PF steps; a longer share in TURNS of them).  The eight partial sums meet in LDS, in pairs.  With a norm in front a wave finds one row's statistics,
// in layernorm_vec_kernel's order, and the fragments are normalised and rounded on their way into the product.
// What bounds it is the trip to memory, as above; no load stands behind a condition here either (rows past either operand's
// re-read its last one: they reach sums that nobody stores).
// WALK: past one workgroup a CU it goes on to the columns of gridDim.x workgroups further, whose weights it asks for under the current
// ones' products; the activations stay in registers, normalised once.
// Steps that a wave may not have, past the rung below in launch_few_k, stand behind uniform branches with nothing on their other side, which
// nobody waits for (asked for in vain: 8 x 4232 -> 1083 6.95 us, 6.3 so).
constexpr int few_steps_sure(int steps, bool LN) {
    return steps == 8 ? 7 : steps == 10 ? 9 : steps == 12 ? (LN ? 9 : 11) : steps == 16 ? 13 : steps == 20 ? 17 : steps == 24 ? 21 : steps == 32 ? 25 : steps == 64 ? 33 : steps;
}
template <int PF, int TURNS, bool LN, bool WALK>
__global__ __launch_bounds__(512) void few_rows_kernel(GemmArgs p, int cols) {
    static_assert(TURNS == 1 || !WALK, "activations in registers");
    constexpr int SURE = few_steps_sure(PF * TURNS, LN);
    constexpr int NW = 8, NA = 5;
    __shared__ float4v red[WALK ? 2 : 1][NW][64];
    __shared__ float lnst[8][2];
    stage_skinny(p);
    const int tid = threadIdx.x, lane = tid & 63, wave = __builtin_amdgcn_readfirstlane(tid >> 6);
    const int row = lane & 15, kq = lane >> 4, nfirst = blockIdx.x * cols, stride = (int)gridDim.x * cols;
    const int steps = (p.K + 31) >> 5, per = (steps + NW - 1) / NW, s0 = wave * per, s1 = min(steps, s0 + per);
    const int mrow = min(row, p.M - 1), wrow = min(row, cols - 1);
    const half_t *const xrow = p.A + (long)mrow * p.ldA;
    struct Cols { u32x4 w[PF]; half_t bias, residual; };
    const int om = (tid >> 4) & 7, oc = tid & 15, omc = min(om, p.M - 1);      // outputs: one of each of the first 128 threads
    auto at = [&](int base, int i) { return min((base + i) * 32 + kq * 8, p.K - 8); };
    auto fetch_w = [&](Cols &c, int n0, auto TURN) {
        constexpr int turn = decltype(TURN)::value;
        const half_t *from = p.B + (long)min(n0 + wrow, p.N - 1) * p.ldB;
#pragma unroll
        for (int i = 0; i < PF; i++)
            if (turn * PF + i < SURE || turn * PF + i < per) c.w[i] = ldg16(from + at(s0 + turn * PF, i));
    };
    auto fetch_out = [&](Cols &c, int n0) {
        const int n = min(n0 + min(oc, cols - 1), p.N - 1);
        const half_t *b = p.bias_mode == MI_BIAS_NONE ? p.B : p.bias + (p.bias_mode == MI_BIAS_COL ? n : omc);
        const half_t *r = p.residual && !p.out_f32 ? p.residual + (long)omc * p.ldY + n : p.B;
        c.bias = *b;
        c.residual = *r;
    };
    u32x4 x[PF], gm[LN ? PF : 1], be[LN ? PF : 1];
    auto fetch_x = [&](auto TURN) {
        constexpr int turn = decltype(TURN)::value;
        const int base = s0 + turn * PF;
#pragma unroll
        for (int i = 0; i < PF; i++) {
            if (turn * PF + i >= SURE && turn * PF + i >= per) continue;
            x[i] = ldg16(xrow + at(base, i));
            if constexpr (LN) {
                gm[i] = ldg16((p.ln_gamma ? p.ln_gamma : p.A) + at(base, i));
                be[i] = ldg16((p.ln_beta ? p.ln_beta : p.A) + at(base, i));
            }
        }
    };
    float mu = 0.0f, rs = 0.0f;
    auto normalise = [&]() {
        if constexpr (LN) {
#pragma unroll
            for (int i = 0; i < PF; i++) {
                const half8v xv = as_half8(x[i]), gv = as_half8(gm[i]), bv = as_half8(be[i]);
                half8v o;
#pragma unroll
                for (int j = 0; j < 8; j++) o[j] = ln_norm1((float)xv[j], mu, rs, p.ln_gamma != nullptr, (float)gv[j], p.ln_beta != nullptr, (float)bv[j]);
                x[i] = __builtin_bit_cast(u32x4, o);
            }
        }
    };
    LnRow<(PF * TURNS + 1) / 2 < 8 ? (PF * TURNS + 1) / 2 : 8> lnrow;      // 512 columns are two steps of eight waves
    if constexpr (LN) lnrow.request(p, min(wave, p.M - 1), lane);
    using I0 = std::integral_constant<int, 0>;
    fetch_x(I0{});
    Cols cur;
    fetch_w(cur, nfirst, I0{});
    fetch_out(cur, nfirst);
    __builtin_amdgcn_sched_barrier(0);
    if constexpr (LN) {
        if (wave < p.M) lnrow.finish(p, lnst, wave, lane);
        __syncthreads();
        mu = lnst[mrow][0];
        rs = lnst[mrow][1];
        normalise();
    }
    float4v acc[NA];
    // five chains, step i of the share in chain i % 5 whatever PF is: short ones keep the error at that of the dot products below five rows
    auto products = [&](const Cols &c, auto TURN) {
        constexpr int turn = decltype(TURN)::value;
        const int base = s0 + turn * PF;
#pragma unroll
        for (int i = 0; i < PF; i++) {
            if (base + i < s1) {                          // uniform
                u32x4 xv = x[i], wv = c.w[i];
                const bool past = (base + i) * 32 + kq * 8 >= p.K;      // in the step that K ends in: neither operand counts there
                const u32x4 z = {0u, 0u, 0u, 0u};
                if ((base + i) * 32 + 32 > p.K) { xv = past ? z : xv; wv = past ? z : wv; }
                float4v &a = acc[(turn * PF + i) % NA];
                a = __builtin_amdgcn_mfma_f32_16x16x32_f16(as_half8(wv), as_half8(xv), a, 0, 0, 0);
            }
        }
    };
    int set = 0;
    for (int nc = nfirst;; nc += stride) {
        Cols nxt;
        const bool more = WALK && p.N - nc > stride;
        if constexpr (WALK) {
            const int nn = more ? nc + stride : p.N - 1;  // (past the end: the last row once more)
            fetch_w(nxt, nn, I0{});
            fetch_out(nxt, nn);
        }
#pragma unroll
        for (int i = 0; i < NA; i++) acc[i] = float4v{0.0f, 0.0f, 0.0f, 0.0f};
        products(cur, I0{});
        auto turn = [&](auto TURN) {
            if constexpr (decltype(TURN)::value < TURNS) {
                fetch_x(TURN);
                fetch_w(cur, nc, TURN);
                normalise();
                products(cur, TURN);
            }
        };
        turn(std::integral_constant<int, 1>{});
        turn(std::integral_constant<int, 2>{});
        turn(std::integral_constant<int, 3>{});
        static_assert(TURNS <= 4, "turns above");
#pragma unroll
        for (int d = 1; d < NA; d *= 2)
#pragma unroll
            for (int i = 0; i + d < NA; i += 2 * d) acc[i] += acc[i + d];
        red[set][wave][lane] = acc[0];
        __syncthreads();
        if (tid < 128 && om < p.M && oc < cols && nc + oc < p.N) {
            const int n = nc + oc;
            float sum[NW];
#pragma unroll
            for (int q = 0; q < NW; q++) sum[q] = reinterpret_cast<const float *>(&red[set][q][(oc >> 2) * 16 + om])[oc & 3];
#pragma unroll
            for (int d = 1; d < NW; d *= 2)
#pragma unroll
                for (int q = 0; q < NW; q += 2 * d) sum[q] += sum[q + d];
            const float t = sum[0] + (p.bias_mode == MI_BIAS_NONE ? 0.0f : (float)cur.bias);
            const long off = (long)om * p.ldY + n;
            if (p.out_f32) reinterpret_cast<float *>(p.Y)[off] = apply_epi(t, p.epi);
            else {
                half_t o = (half_t)apply_epi((float)(half_t)t, p.epi);
                if (p.residual) o = (half_t)((float)o + (float)cur.residual);
                reinterpret_cast<half_t *>(p.Y)[off] = o;
            }
        }
        if constexpr (!WALK) break;
        else {
            if (!more) break;
            cur = nxt;
            set ^= 1;                                     // (a wave two turns ahead of a reader has passed that reader's barrier)
        }
    }
}

// The same product with the activations in registers instead of LDS, for one or two rows of K <= 1536 without a norm: a lane's
// weight chunks sit at k = 8 lane + 512 i, so it needs exactly those chunks of every activation row and asks for
// them itself (the rows come from the L2: every wave of the launch reads the same few KB).  No staging, no barrier: one trip to
// memory, the dot products, one wave reduction and a store.
template <int MT, int PF>
__global__ __launch_bounds__(256) void skinny_fk_reg_kernel(GemmArgs p) {
    stage_skinny(p);
    const int lane = threadIdx.x & 63, wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
    const int n = blockIdx.x * 4 + wave;
    u32x4 x[MT][PF], w[1][PF];
#pragma unroll
    for (int m = 0; m < MT; m++)
#pragma unroll
        for (int i = 0; i < PF; i++) x[m][i] = ldg16(p.A + (long)min(m, p.M - 1) * p.ldA + min(lane * 8 + 512 * i, p.K - 8));
    fk_request(p, w, n, lane);
    FkOut<MT, 1> out;
    out.request(p, n, lane);
    float acc[MT] = {};
#pragma unroll
    for (int i = 0; i < PF; i++)
        if (lane * 8 + 512 * i < p.K) {
#pragma unroll
            for (int m = 0; m < MT; m++) acc[m] = fk_dot(w[0][i], x[m][i], acc[m]);
        }
    float mine = 0.0f;
#pragma unroll
    for (int m = 0; m < MT; m++) {
        const float sres = wave_sum(acc[m]);
        if (lane == m) mine = sres;
    }
    out.store(p, mine, n, lane);
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

// Whether [K][F] weights run as 32 x 32 tiles with K over the waves of a workgroup (gemm_deep_kernel) instead of K-slices and the launch
// that sums them.  The tiles are one launch and one trip to memory, their products on the matrix cores; the slices have more loads in
// flight where a large weight comes from memory.  us, slices | tiles: 384 -> 1536 one row 6.1 | 3.4, eight 9.2 | 3.5; 64 -> 128 4.2 | 3.2,
// 7.4 | 3.2; 1280 -> 5120 four rows 8.2 | 4.7, from memory 10.0 | 8.5, and one row 6.2 | 6.0, from memory 8.2 | 9.3: hence the megabytes.
// With a norm in front the rows are normalised into the planes' memory first, by the norm's own kernel, for the bits of the two calls:
// 384 -> 1536 7.2 | 5.3, 11.4 | 5.5.  That is slower for one or two rows past K = 768 (1032 -> 136 6.4 | 7.6; 768 -> 768 7.1 | 6.2).  Error
// against 64 bits (fp32 results, 64 <= K <= 1280): 0.76 to 0.96 of the slices'; past that it is theirs that is smaller (1536 -> 384
// 8.6e-8 | 1.0e-7), so they stay.
bool kn_on_tiles(int64_t T, int64_t K, int64_t F, size_t planes) {
    if (K > (T <= 2 ? 768 : 1280) || planes < (size_t)(T * K) * sizeof(half_t)) return false;
    const double mb = 2e-6 * (double)K * (double)F, rows = T <= 1 ? 0.0 : T <= 2 ? 0.4 : T <= 4 ? 1.3 : 3.4;
    return mi_deep_us(T, K, F) + 0.25 * std::min(mb, 16.0) < 5.9 + rows + 0.15 * mb + 1.2e-6 * (double)planes;
}

// few_rows_kernel from five rows on.  us at four rows on the kernels above, at eight on the matrix cores: 1280 -> 5120 5.2 and 6.6, 4096 -> 1024
// 5.7 and 7.2, 5120 -> 1280 7.6 and 8.4, 1280 -> 51866 27.3 and 26.2, 1536 -> 384 3.2 and 3.8 (the kernels above hold four rows at most).
constexpr int FEW_ROWS_MIN = 5;

template <int PF, int TURNS, bool LN>
void launch_few(const GemmArgs &a, hipStream_t st) {
    const int cols = ceil_div(a.N, 16) * 2 <= mi_num_cus() ? 8 : 16;
    const int64_t wgs = ceil_div(a.N, cols);
    // Past one workgroup a CU the registers of a norm (160 and up) let no second one in, and without a norm the activations are read once a
    // workgroup: eight rows of 1280 -> 51866 30.5 us with a workgroup for every sixteen columns, 26.2 walking (behind a norm 70.5 and 28.4).
    // Two workgroups a CU where the registers allow it and there are turns enough (384 -> 51866 13.6 | 10.0, -> 9000 3.9 | 4.0); from
    // K = 1281 on none walks (2048 -> 8192 9.5 | 10.2).
    if constexpr (TURNS == 1 && PF <= 5) {
        const int64_t cus = mi_num_cus(), two = PF <= (LN ? 2 : 3) && wgs > 4 * cus ? 2 : 1;
        if (wgs > cus) {
            hipLaunchKernelGGL((few_rows_kernel<PF, 1, LN, true>), dim3((unsigned)(cus * two)), dim3(512), 0, st, a, cols);
            return;
        }
    }
    hipLaunchKernelGGL((few_rows_kernel<PF, TURNS, LN, false>), dim3((unsigned)wgs), dim3(512), 0, st, a, cols);
}

// By the 32-deep steps that each of the eight waves takes: K <= 16 384, as the caller's bound on LDS says, behind a norm half of it.
// Steps past a wave's share cost the loads' issue, and registers decide the waves in flight, so a rung is its kernel (few_steps_sure: what
// lies between two).  us of eight rows -> 1280, weights from memory, on its rung | with all steps of the next asked for: K 512 2.75 | 2.98, 768 3.02 | 3.26, 1024 3.28 | 3.51, 1280 3.52 | 3.76, 1536 3.78 |
// 4.38, 2048 4.42 | 4.90, 2560 4.92 | 5.56, 3072 5.58 | 6.72, 4096 6.96 | 7.79, 5120 7.94 | 9.20, 6144 9.28 | 11.4; behind a norm 512 3.72 |
// 4.04, 768 4.42 | 4.64, 1024 4.73 | 5.29, 1280 5.77 | 6.15, 1536 6.32 | 7.18, 2048 7.68 | 8.46, 3072 9.15 | 11.0, 4096 11.7 | 13.2, 5120 17.1 | 17.6,
// 6144 19.0 | 20.1 (ten steps at once for K up to 2560 there: 9.01, 8.95 in two rounds of six).
int launch_few_k(const GemmArgs &a, hipStream_t st) {
    const int64_t per = ceil_div(ceil_div(a.K, 32), 8);
    if (per > (a.ln_on ? 32 : 64)) return MI_DECLINE_EXTENT;
    if (a.ln_on) {
        if (per <= 2)       launch_few<2, 1, true>(a, st);
        else if (per <= 3)  launch_few<3, 1, true>(a, st);
        else if (per <= 4)  launch_few<4, 1, true>(a, st);
        else if (per <= 5)  launch_few<5, 1, true>(a, st);
        else if (per <= 6)  launch_few<6, 1, true>(a, st);
        else if (per <= 8)  launch_few<8, 1, true>(a, st);
        else if (per <= 12) launch_few<6, 2, true>(a, st);
        else if (per <= 16) launch_few<8, 2, true>(a, st);
        else if (per <= 20) launch_few<10, 2, true>(a, st);
        else if (per <= 24) launch_few<8, 3, true>(a, st);
        else                launch_few<8, 4, true>(a, st);
    } else {
        if (per <= 2)       launch_few<2, 1, false>(a, st);
        else if (per <= 3)  launch_few<3, 1, false>(a, st);
        else if (per <= 4)  launch_few<4, 1, false>(a, st);
        else if (per <= 5)  launch_few<5, 1, false>(a, st);
        else if (per <= 6)  launch_few<6, 1, false>(a, st);
        else if (per <= 8)  launch_few<8, 1, false>(a, st);
        else if (per <= 10) launch_few<10, 1, false>(a, st);
        else if (per <= 12) launch_few<12, 1, false>(a, st);
        else if (per <= 16) launch_few<16, 1, false>(a, st);
        else if (per <= 20) launch_few<20, 1, false>(a, st);
        else if (per <= 24) launch_few<12, 2, false>(a, st);
        else if (per <= 32) launch_few<16, 2, false>(a, st);
        else                launch_few<16, 4, false>(a, st);
    }
    return MI_OK;
}

template <int MT, int PF>
void launch_fk(const GemmArgs &a, hipStream_t st) {
    const size_t lds = (size_t)MT * a.K * sizeof(half_t);
    const int64_t cus = mi_num_cus();
    auto go = [&](auto R_, auto LN_, int64_t cap) {
        constexpr int R = decltype(R_)::value;
        const int64_t wgs = ceil_div(a.N, 4 * R);
        hipLaunchKernelGGL((skinny_fk_kernel<MT, PF, R, decltype(LN_)::value>), dim3((unsigned)(wgs < cap ? wgs : cap)), dim3(256), lds, st, a);
    };
    using std::integral_constant;
    if constexpr (PF > 3) {                               // (a long row fills the registers by itself)
        if (a.ln_on) go(integral_constant<int, 1>{}, std::true_type{}, 8 * cus);
        else go(integral_constant<int, 1>{}, std::false_type{}, 8 * cus);
    } else {
        // Up to 8192 columns every group has its wave.  A wider output -- a vocabulary -- is walked by two or three workgroups a CU, three columns a
        // wave and turn: 1280 -> 51866 at one, two and four rows 24.3, 25.1, 27.3 us (30.5, 32.1, 35.0 with a column a wave, eight
        // workgroups a CU and the next column asked for behind a branch), behind a norm 24.0, 24.6, 27.6 (31.9, 34.4, 38.4).
        if (!a.ln_on && a.N <= 8192) {
            if constexpr (MT <= 2) hipLaunchKernelGGL((skinny_fk_reg_kernel<MT, PF>), dim3((unsigned)ceil_div(a.N, 4)), dim3(256), 0, st, a);
            else go(integral_constant<int, 1>{}, std::false_type{}, 8 * cus);
        } else if (!a.ln_on) {
            go(integral_constant<int, 3>{}, std::false_type{}, 3 * cus);
        } else switch (a.N <= 8192 ? ceil_div(a.N, 4 * cus) : 3) {
            case 0: case 1: case 2: go(integral_constant<int, 2>{}, std::true_type{}, 2 * cus); break;
            case 3: go(integral_constant<int, 3>{}, std::true_type{}, 2 * cus); break;
            case 4: go(integral_constant<int, 4>{}, std::true_type{}, 2 * cus); break;
            default: go(integral_constant<int, 5>{}, std::true_type{}, 2 * cus); break;
        }
    }
}

template <int MT, int PF>
int raise_fk() {
    auto up = [](auto kern) { return raise_lds(kern, (int)SKINNY_FK_LDS_MAX); };
    return up(skinny_fk_kernel<MT, PF, 1, false>) | up(skinny_fk_kernel<MT, PF, 1, true>);
}

// By the 512-column chunks of a row.  us of one row -> 1280 | four rows behind a norm -> 5120, weights from memory, on its rung and on the
// next: K 512 2.19, 2.32 | 4.61, 4.94; 1024 2.31, 2.40 | 5.48, 5.99; 1536 2.44, 3.10 | 7.4, 12.8; 3072 3.24, 3.38 | 17.2, 18.0; 4096 3.49,
// 3.81 | 21.8, 22.8; 5120 4.93, 5.09 | 27.1, 35.2.
template <int MT>
void launch_fk_k(const GemmArgs &a, hipStream_t st) {
    if (a.K <= 512) launch_fk<MT, 1>(a, st);
    else if (a.K <= 1024) launch_fk<MT, 2>(a, st);
    else if (a.K <= 1536) launch_fk<MT, 3>(a, st);
    else if (a.K <= 3072) launch_fk<MT, 6>(a, st);
    else if (a.K <= 4096) launch_fk<MT, 8>(a, st);
    else if (a.K <= 5120) launch_fk<MT, 10>(a, st);
    else launch_fk<MT, 12>(a, st);
}

}  // namespace

int mi_skinny_splits(int64_t K, int64_t F) { return (int)ceil_div(K, skinny_kper(K, F)); }

static size_t planes_bytes(int64_t T, int64_t K, int64_t F) { return (size_t)mi_skinny_splits(K, F) * T * F * sizeof(float); }
int mi_skinny_slices(int64_t T, int64_t K, int64_t F, int64_t ldA, int64_t ldB) {
    return mi_deep_takes(ldA, ldB) && kn_on_tiles(T, K, F, planes_bytes(T, K, F)) ? 1 : mi_skinny_splits(K, F);
}

int mi_skinny_launch(const GemmArgs &a, bool b_kn, void *ws, size_t ws_bytes, hipStream_t st) {
    if (b_kn) {
        const int kper = skinny_kper(a.K, a.N), nsplit = (int)ceil_div(a.K, kper);
        const size_t need = planes_bytes(a.M, a.K, a.N);
        if (!ws || ws_bytes < need || !aligned_to(ws, 256)) return MI_DECLINE_WORKSPACE;
        if (mi_deep_takes(a.ln_on ? a.K : a.ldA, a.ldB) && kn_on_tiles(a.M, a.K, a.N, need)) {
            GemmArgs t = a;
            if (a.ln_on) {
                t.ln_on = 0; t.A = reinterpret_cast<const half_t *>(ws); t.ldA = a.K;
                const int rc = mi_internal_layernorm(ws, nullptr, nullptr, a.A, a.ldA, a.ln_gamma, a.ln_beta, a.K, a.M, a.ln_eps, st);
                if (rc != MI_OK) return rc;
            }
            return mi_deep_launch(t, true, true, 1, st);
        }
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
            const int rc = launch_few_k(a, st);
            if (rc != MI_OK) return rc;
        } else if (mt == 1) launch_fk_k<1>(a, st);
        else if (mt == 2) launch_fk_k<2>(a, st);
        else launch_fk_k<4>(a, st);
    }
    return hipGetLastError() == hipSuccess ? MI_OK : MI_ERROR_LAUNCH;
}

int mi_skinny_init() {
    int bad = 0;
    bad |= raise_fk<1, 6>() | raise_fk<1, 8>() | raise_fk<1, 10>() | raise_fk<1, 12>();
    bad |= raise_fk<2, 6>() | raise_fk<2, 8>() | raise_fk<2, 10>() | raise_fk<2, 12>();
    bad |= raise_fk<4, 6>() | raise_fk<4, 8>() | raise_fk<4, 10>() | raise_fk<4, 12>();
    return bad;
}
