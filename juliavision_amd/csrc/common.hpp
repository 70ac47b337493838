// Shared device/host helpers for the gfx950 kernels.
#pragma once
#include <hip/hip_runtime.h>
#include <stdint.h>
#include "extents.hpp"
#include "../../include/mi355dnn.h"

typedef _Float16 half_t;
typedef _Float16 half2v __attribute__((ext_vector_type(2)));
typedef _Float16 half4v __attribute__((ext_vector_type(4)));
typedef _Float16 half8v __attribute__((ext_vector_type(8)));
typedef float float4v __attribute__((ext_vector_type(4)));
typedef float float2v __attribute__((ext_vector_type(2)));
typedef float float16v __attribute__((ext_vector_type(16)));
typedef uint32_t u32x4 __attribute__((ext_vector_type(4)));
typedef uint32_t u32x2 __attribute__((ext_vector_type(2)));
typedef short short4v __attribute__((ext_vector_type(4)));
typedef short short8v __attribute__((ext_vector_type(8)));

#define MI_DEVICE static __device__ __forceinline__

MI_DEVICE u32x4 ldg16(const half_t *p) { return *reinterpret_cast<const u32x4 *>(p); }
MI_DEVICE u32x2 ldg8(const half_t *p) { return *reinterpret_cast<const u32x2 *>(p); }

// lo16(x) | lo16(y) << 16   and   hi16(x) | hi16(y) << 16
MI_DEVICE uint32_t pack_lo(uint32_t x, uint32_t y) { return __builtin_amdgcn_perm(y, x, 0x05040100u); }
MI_DEVICE uint32_t pack_hi(uint32_t x, uint32_t y) { return __builtin_amdgcn_perm(y, x, 0x07060302u); }

// x / d and what is left, with recip = recip_of(d) from the host: the product's upper half is the quotient or one less, for every 32-bit
// dividend, and no case needs a branch.  A division by a value that arrives with the launch is some thirty instructions.
MI_DEVICE unsigned divide(unsigned x, unsigned d, unsigned recip, unsigned &left) {
    unsigned q = __umulhi(x, recip), r = x - q * d;
    const bool up = r >= d;
    q += up ? 1u : 0u;
    left = r - (up ? d : 0u);
    return q;
}
static inline unsigned recip_of(int64_t d) { return (unsigned)(0xffffffffll / d); }

MI_DEVICE half8v as_half8(u32x4 v) { return __builtin_bit_cast(half8v, v); }

// Lane exchanges without the LDS crossbar.  lane_xor<O>(v) is v of lane (lane ^ O) for O = 1, 2, 4, 8: data-parallel
// primitives riding on the consuming VALU instruction (quad permutes, a rotation by 8 inside each row of 16, and for 4
// the mirror of 8 lanes followed by the mirror of 4: lane ^ 7 ^ 3).  Across rows gfx950 has v_permlane16_swap /
// v_permlane32_swap, which exchange the odd rows of one register with the even rows of another: from two copies of v
// they leave (even rows twice, odd rows twice), whose sum or maximum is op(v[lane], v[lane ^ 16]) in every lane.
// wave_sum / wave_max are the butterflies over 32, 16, 8, 4, 2, 1 built from these: the pairs, the order and therefore
// the bits are those of the same butterfly written with __shfl_xor (six ds_bpermute round trips).
template <int CTRL>
MI_DEVICE float dpp_mov(float v) { return __builtin_bit_cast(float, __builtin_amdgcn_update_dpp(0, __builtin_bit_cast(int, v), CTRL, 0xF, 0xF, true)); }
template <int O>
MI_DEVICE float lane_xor(float v) {
    static_assert(O == 1 || O == 2 || O == 4 || O == 8, "inside a row of 16 lanes");
    if constexpr (O == 1) return dpp_mov<0xB1>(v);             // quad_perm [1,0,3,2]
    else if constexpr (O == 2) return dpp_mov<0x4E>(v);        // quad_perm [2,3,0,1]
    else if constexpr (O == 4) return dpp_mov<0x1B>(dpp_mov<0x141>(v));   // row_half_mirror, then quad_perm [3,2,1,0]
    else return dpp_mov<0x128>(v);                              // row_ror:8
}
// (x, y) <- (even 32-lane halves of both, odd halves of both); the instruction is written out because the builtin's
// second result is miscompiled when both operands hold the same value.
MI_DEVICE void swap_rows32(float &x, float &y) { asm volatile("s_nop 1\n\tv_permlane32_swap_b32 %0, %1\n\ts_nop 1" : "+v"(x), "+v"(y)); }
MI_DEVICE void swap_rows16(float &x, float &y) { asm volatile("s_nop 1\n\tv_permlane16_swap_b32 %0, %1\n\ts_nop 1" : "+v"(x), "+v"(y)); }
MI_DEVICE float wave_sum(float a) {
    float x = a, y = a;
    swap_rows32(x, y); a = x + y;
    x = a; y = a;
    swap_rows16(x, y); a = x + y;
    a += lane_xor<8>(a);
    a += lane_xor<4>(a);
    a += lane_xor<2>(a);
    a += lane_xor<1>(a);
    return a;
}
MI_DEVICE float wave_max(float a) {
    float x = a, y = a;
    swap_rows32(x, y); a = fmaxf(x, y);
    x = a; y = a;
    swap_rows16(x, y); a = fmaxf(x, y);
    a = fmaxf(a, lane_xor<8>(a));
    a = fmaxf(a, lane_xor<4>(a));
    a = fmaxf(a, lane_xor<2>(a));
    a = fmaxf(a, lane_xor<1>(a));
    return a;
}

// Abramowitz & Stegun 7.1.26 in fp32: the same expression as the reference's
// `erf` (DNNKernels/src/ops.jl:161-169), so a folded gelu is the graph's gelu.
MI_DEVICE float erf_as(float x) {
    float a = fabsf(x);
    float t = __builtin_amdgcn_rcpf(1.0f + 0.3275911f * a);
    float y = 1.0f - (((((1.061405429f * t - 1.453152027f) * t) + 1.421413741f) * t - 0.284496736f) * t + 0.254829592f) * t * __expf(-a * a);
    return x < 0.0f ? -y : y;
}
// geluexact (DNNKernels/src/ops.jl:1665-1669) = 0.5 v (1 + erf(v / sqrt 2)) with the erf above, in as few vector instructions
// as there are (the GEMM store is bound by them: 32 768 outputs per workgroup).  With u = |v|, t = 1 / (1 + p u / sqrt 2) and
// q = 0.5 P(t) exp(-v^2 / 2):
//   v >= 0:  0.5 v (2 - P e) = v - v q        v < 0:  0.5 v (P e) = v q        both:  max(v, 0) - u q,
// Same polynomial, same coefficients; the difference from the textbook order is rounding in the last fp32 place (and, for v < -3,
// none of the cancellation in 1 - (1 - P e)), far below the fp16 result's resolution.  u 2^(-u^2 log2(e) / 2) lies in [0, 0.61]: the
// clamp, a modifier of the product, changes nothing but infinity times 0, so that v = +inf gives +inf as the reference's
// expression does (t is 0 there), v = -inf 0 (the reference: -inf * 0 = NaN).  NaN stays NaN by way of t.  Products with u are
// written as fused ones: of an fp16 u they take the conversion in.
MI_DEVICE float gelu_erf_of(float u, float above) {      // |v|, max(v, 0)
    const float t = __builtin_amdgcn_rcpf(fmaf(u, 0.3275911f * 0.70710678118654752440f, 1.0f));
    float pl = fmaf(0.5f * 1.061405429f, t, -0.5f * 1.453152027f);
    pl = fmaf(pl, t, 0.5f * 1.421413741f);
    pl = fmaf(pl, t, -0.5f * 0.284496736f);
    pl = fmaf(pl, t, 0.5f * 0.254829592f);
    pl *= t;
    const float e = __builtin_amdgcn_exp2f(fmaf(u, u, 0.0f) * (-0.5f * 1.44269504088896340736f));
    return fmaf(-pl, __builtin_amdgcn_fmed3f(fmaf(u, e, 0.0f), 0.0f, 1.0f), above);
}
MI_DEVICE float gelu_erf(float v) { return gelu_erf_of(fabsf(v), fmaxf(v, 0.0f)); }
// ops.jl:1665-1669 (geluexact), 1677-1682 (gelutanh), 1683 (relu_epi)
MI_DEVICE float apply_epi(float v, int epi) {
    switch (epi) {
    case MI_EPI_GELU_ERF: return gelu_erf(v);
    case MI_EPI_GELU_TANH: return 0.5f * v * (1.0f + tanhf(0.7978845608028654f * (v + 0.044715f * v * v * v)));
    case MI_EPI_RELU: return fmaxf(v, 0.0f);
    default: return v;
    }
}

template <int EPI>
MI_DEVICE float apply_epi_c(float v) {
    if constexpr (EPI == MI_EPI_GELU_ERF) return gelu_erf(v);
    else if constexpr (EPI == MI_EPI_GELU_TANH) return 0.5f * v * (1.0f + tanhf(0.7978845608028654f * (v + 0.044715f * v * v * v)));
    else if constexpr (EPI == MI_EPI_RELU) return fmaxf(v, 0.0f);
    else return v;
}

// Eight fp16 values at once, the bits those of apply_epi_c on each: max(v, 0) is half an instruction a value in fp16, |v| none.
// 13.6 vector instructions a value for the erf-GELU, two of them transcendental, where a value at a time took 15.6 (1500 x 1280 ->
// 5120: 24.6 -> 23.8 us; over every fp16 value the same error against 64 bits to seven digits).
template <int EPI>
MI_DEVICE half8v apply_epi8(half8v v) {
    if constexpr (EPI == MI_EPI_GELU_ERF) {
        const half8v above = __builtin_elementwise_max(v, half8v{});
#pragma unroll
        for (int e = 0; e < 8; e++) v[e] = (half_t)gelu_erf_of((float)__builtin_fabsf16(v[e]), (float)above[e]);
    } else if constexpr (EPI != MI_EPI_NONE) {
#pragma unroll
        for (int e = 0; e < 8; e++) v[e] = (half_t)apply_epi_c<EPI>((float)v[e]);
    }
    return v;
}

// One layer-normalised element, rounded to fp16: shared by the layer-norm kernels and the GEMV that folds
// the norm into its prologue, so that the two produce the same bits.
MI_DEVICE half_t ln_norm1(float x, float mu, float r, bool has_g, float g, bool has_b, float b) {
    float y = (x - mu) * r;
    if (has_g) y *= g;
    if (has_b) y += b;
    return (half_t)y;
}

static inline bool aligned_to(const void *p, size_t a) { return (reinterpret_cast<uintptr_t>(p) % a) == 0; }
// NaN by its bits: the build tells the compiler that no NaNs occur, which folds comparisons with one away.
static inline bool is_nan_arg(float x) { uint32_t u; __builtin_memcpy(&u, &x, 4); return (u & 0x7fffffffu) > 0x7f800000u; }

// Largest image, in halves, of the gather below: gemm_ring_kernel's offsets into it are 32-bit byte offsets, raised by up to 3072.
constexpr int64_t MI_PATCH_IMAGE_MAX = INT32_MAX - 1536;
// Implicit-GEMM convolution over a zero-padded channels-last copy xp[img][Hp][Wp][C] of the input: how gemm_ring_kernel and
// gemm_deep_kernel find their [N][K] operand (row n = output pixel (oh, ow), K ordered (kh, kw, ci) with ci fastest) in it.  Sixteen bytes of a
// row are eight channels of one tap, at an offset from the pixel's origin that is the same for every pixel.
struct ConvGather {
    const half_t *xp;      // nullptr = ordinary GEMM
    long img;              // elements per image
    int C, OW, KW;
    int pix_y, pix_x;      // elements between the origins of neighbouring output rows and columns: sy Wp C, sx C
    int tap_y, tap_x;      // and between neighbouring taps: dy Wp C, dx C
    unsigned div_C, div_OW, div_KW;      // recip_of
};

// Implicit-GEMM convolution over a channels-last input x[N][H][W][C]: how the GEMM finds its [M][K] operand
// (the patch matrix: row m = output pixel (n, oh, ow), K ordered (kh, kw, ci) with ci fastest) in x itself.
// A 64-deep tile is 64 consecutive channels of one tap, i.e. 128 contiguous bytes of x per row, at an offset
// from the row's pixel that is the same for every row; rows whose tap falls outside the image read zeros.
struct NhwcGather {
    const half_t *x;       // nullptr = ordinary GEMM
    int H, W, C, OH, OW;
    int sx, sy, px, py, dx, dy, KW;
    int cpt;               // 64-channel tiles per tap: C / 64
    int split;             // 1: the launch's planes are K-slices
};

// True once mi_init has run successfully on this process (defined in gemm.hip).
bool mi_ready();
int mi_num_cus();
// Planning for a device other than the current one (mi_*_plan_caps): between begin and end, on this thread,
// mi_num_cus() and mi_plan_mfma() answer for caps (the six values of mi_device_caps); caps == nullptr changes nothing.
bool mi_plan_mfma();
void mi_plan_caps_begin(const int64_t *caps);
void mi_plan_caps_end();
// True if the current device deals workgroups to its XCDs round robin by workgroup id (ids that differ by a multiple
// of 8 share an L2), as a probe launch at mi_init showed; kernels whose workgroups exchange data through one L2 ask.
bool mi_xcd_round_robin();
int mi_sdpa_init();
// Y[M x N] = A[M x K] . B (+bias) (+ residual, fp16, addressed like Y with batch stride sY + dres) with B either [K][NB-padded N] (b_kn) or [N][K]; defined in gemm.hip.
int mi_internal_gemm(void *Y, const void *A, const void *B, const void *bias, int M, int N, int NB, int K,
                     long ldY, long ldA, long ldB, int b_kn, int bias_mode, int epi, int out_f32,
                     long nbatch, long sY, long sA, long sB, void *ws, size_t ws_bytes, hipStream_t st,
                     const ConvGather *gather = nullptr, const NhwcGather *agather = nullptr, const void *residual = nullptr, long dres = 0);
// Workspace bytes such a call needs (fp32 planes when it splits K); T > 8 rows.
size_t mi_internal_gemm_workspace(int64_t T, int64_t K, int64_t F, int64_t nbatch);
// What such a call is estimated to take, in microseconds.
int mi_internal_layernorm(void *out, float *mean, float *rstd, const void *a, int64_t lda, const void *gamma, const void *beta, int64_t C, int64_t groups, float eps, void *stream);
double mi_internal_patch_gemm_us(int64_t T, int64_t K, int64_t F, int64_t nbatch);      // B a ConvGather: on the kernel that is estimated to be faster
int mi_internal_patch_kernel(int64_t T, int64_t K, int64_t F, int64_t nbatch);          // that kernel: an mi_gemm_kernel
double mi_internal_gemm_us(int64_t T, int64_t K, int64_t F, int64_t nbatch);
