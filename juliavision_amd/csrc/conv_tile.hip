// Convolution for gfx950 in one launch, [N][Cin][H][W] -> [N][Cout][OH][OW], one group, any kernel, stride, padding and
// dilation: an implicit GEMM over K = (ci, kh, kw) in the order the weights lie in memory.
//
// A workgroup owns a TH x TW rectangle of output pixels (32 a wave) times 32 TCO output channels.  Per chunk of CC input
// channels it stages the input patch those pixels see (rows padded with zeros, 16-byte pieces) and the chunk's weights
// (contiguous runs of CC KH KW halves per output channel) in LDS.  The pixel operand of the MFMA is assembled from the
// patch: a lane is a pixel, and its eight consecutive k are eight two-byte LDS reads at the pixel's origin plus an offset
// from a table (the same for all pixels; an entry per k of a chunk).  Every assembled fragment meets TCO weight fragments.
// The next chunk's pieces are in flight in registers during this chunk's MFMAs.
//
// The im2col matrix (K / CC times the input), its GEMM's two reads of it and the launches between are gone: 1024 x 1024 x 3 ->
// 144, 7 x 7 stride 4, 50.9 -> 15.1 us (floor 4.8).  Bound by its own serial chain, there one chunk, all of it staged before the
// first product: of 25 000 clocks in the kernel 12 000 are the staging (two batches of loads, each a trip to memory, and at two-byte
// addresses four times the vector-memory time of aligned ones), 6400 the products and the pixel operand's two-byte reads, 6500 the store.
#include "conv_common.hpp"
#include <type_traits>

using namespace conv_tile;

namespace {

typedef unsigned short u16x8 __attribute__((ext_vector_type(8)));

// The plan, the problem, and the kernel's divisions as multiplications (divide): some thirty instructions each otherwise, four a piece.
struct TileConv : TilePlan {
    ConvArgs a;
    unsigned div_x, div_taps, div_kw, div_tw, div_pc, div_pr, div_wp;
};

// PW waves side by side over pixels, KG groups of them over the steps of a chunk, TCO x 32 output channels each.
// WP, PP: weight and patch pieces a thread carries in registers for the next chunk.
// CHUNKS: 1 a single chunk, 2 several, each a kernel of its own: together their conditions did not fit the scalar registers.  0 either,
// for rows of the image or of the weights too short for a 16-byte piece, read by element.
template <int PW, int KG, int TCO, int CHUNKS>
__global__ __launch_bounds__(PW *KG * 64) void conv_tile_kernel(TileConv t) {
    constexpr bool ELEM = CHUNKS == 0;
    constexpr int NT = PW * KG * 64, CO = 32 * TCO, WP = TCO > 2 ? 6 : 5, PP = 3;
    extern __shared__ __align__(16) char smem[];
    const ConvArgs &a = t.a;
    const int tid = threadIdx.x, lane = tid & 63, wave = __builtin_amdgcn_readfirstlane(tid >> 6), pw = wave % PW, kg = wave / PW;
    const int taps = a.KH * a.KW, CRS = a.Cin * taps;
    const int HiWi = a.Hi * a.Wi;
    auto over = [](int v, int d, unsigned recip, int &left) { unsigned l; const int q = (int)divide((unsigned)v, (unsigned)d, recip, l); left = (int)l; return q; };
    int tx;
    const int ty = over(blockIdx.x, t.tiles_x, t.div_x, tx);
    const int oy0 = ty * t.TH, ox0 = tx * t.TW, co0 = blockIdx.y * CO;
    const half_t *x = a.x + (long)blockIdx.z * a.Cin * HiWi;
    const int iy0 = oy0 * a.sy - a.py, ix0 = ox0 * a.sx - a.px;
    const int xa = ix0 & ~7;                              // the patch starts on a multiple of eight image columns
    unsigned short *tab = reinterpret_cast<unsigned short *>(smem + t.tab_off);
    const int zero_at = t.CC * t.PR * t.PCL;            // eight halves behind the patch stay zero

    // k of a chunk -> offset in the patch (halves); steps end on a multiple of 16 past kc: those entries point at the zeros
    for (int k = tid; k < t.ksteps * 16; k += NT) {
        int off = zero_at;
        if (k < t.kc) {
            int r, kw;
            const int ci = over(k, taps, t.div_taps, r), kh = over(r, a.KW, t.div_kw, kw);
            off = (ci * t.PR + kh * a.dy) * t.PCL + kw * a.dx;
        }
        tab[k] = (unsigned short)off;
    }

    // Eight halves of which the first `gone` are dropped and zeros follow: what a load that was moved back to stay inside its
    // row turns into.
    auto shifted = [](u32x4 v, int gone) {
        const uint64_t lo = (uint64_t)v[0] | (uint64_t)v[1] << 32, hi = (uint64_t)v[2] | (uint64_t)v[3] << 32;
        const int b = 16 * gone;                         // 0 .. 112
        const uint64_t l = b >= 64 ? hi >> (b - 64) : b ? lo >> b | hi << (64 - b) : lo, h = b >= 64 ? 0 : hi >> b;
        const u32x4 r = {(uint32_t)l, (uint32_t)(l >> 32), (uint32_t)h, (uint32_t)(h >> 32)};
        return r;
    };
    const bool narrow = ELEM && a.Wi < 8, short_w = ELEM && weights_by_element(t.kc, CRS);      // uniform
    const u32x4 zero4 = {0u, 0u, 0u, 0u};
    // A 16-byte piece: where it lies in memory (halves from the chunk's start) and in the stage (bytes); k or channel of the
    // chunk it starts at; how many of its halves a load moved back to stay inside the row drops.
    struct Piece { int src, dst, lim, gone; bool have; };
    // Patch: row `row` of channel `ci`, image columns ix .. ix + 7 (ix a multiple of 8: never cut at the left).
    auto patch_of = [&](int c) {
        int j, row;
        const int q = over(c, t.PC8, t.div_pc, j), ci = over(q, t.PR, t.div_pr, row), iy = iy0 + row, ix = xa + 8 * j;
        Piece p;
        p.have = c < t.patch_pieces && (unsigned)iy < (unsigned)a.Hi && (unsigned)ix < (unsigned)a.Wi;
        p.gone = p.have && !narrow ? max(0, ix + 8 - a.Wi) : 0;
        p.src = p.have ? ci * HiWi + iy * a.Wi + ix - p.gone : 0;
        p.dst = (q * t.PCL + 8 * j) * 2;
        p.lim = ci;
        return p;
    };
    auto weight_of = [&](int c) {
        int j;
        const int co = over(c, t.wpieces, t.div_wp, j);
        Piece p;
        p.have = c < t.weight_pieces && 8 * j < t.kc;
        p.src = p.have ? min(co0 + co, a.Cout - 1) * CRS + 8 * j : 0;      // rows past Cout repeat the last one: their results are never stored
        p.dst = (co * t.WLD + 8 * j) * 2;
        p.lim = 8 * j;
        p.gone = 0;
        return p;
    };
    // A load and what it turns into (`patch_fixed`, `weight_fixed`, once it is used) are apart, and no load stands behind a condition: where
    // the two sides of one meet the compiler waits for it, and the pieces of a chunk came one trip to memory after the other.
    // What does not exist -- outside the image, past the chunk or past Cin -- reads the tensor's first piece.
    auto patch_in = [&](const Piece &p, int c0) { return p.have && c0 + p.lim < a.Cin; };
    auto weight_left = [&](const Piece &p, int c0) { return p.have ? weight_end(t.kc, CRS, c0 * taps) - p.lim : 0; };
    auto patch_load = [&](const Piece &p, int c0) {
        u32x4 v = zero4;
        if (narrow) {
            half8v h = as_half8(v);
            if (patch_in(p, c0)) {
                const half_t *s = x + (long)c0 * HiWi + p.src;
#pragma unroll
                for (int e = 0; e < 8; e++) if (e < a.Wi) h[e] = s[e];      // ix is 0
            }
            return __builtin_bit_cast(u32x4, h);
        }
        const half_t *s = patch_in(p, c0) ? x + (long)c0 * HiWi + p.src : x;
        __builtin_memcpy(&v, s, 16);
        return v;
    };
    auto patch_fixed = [&](u32x4 v, const Piece &p, int c0) {
        if (narrow) return v;
        if (__any(p.gone)) v = shifted(v, p.gone);
        return patch_in(p, c0) ? v : zero4;
    };
    auto weight_load = [&](const Piece &p, int c0) {
        const int left = weight_left(p, c0);
        u32x4 v = zero4;
        if (short_w) {
            half8v h = as_half8(v);
            if (left > 0) {
                const half_t *s = a.w + c0 * taps + p.src;
#pragma unroll
                for (int e = 0; e < 8; e++) if (e < left) h[e] = s[e];
            }
            return __builtin_bit_cast(u32x4, h);
        }
        const half_t *s = left > 0 ? a.w + c0 * taps + p.src - weight_back(left) : a.w;
        __builtin_memcpy(&v, s, 16);
        return v;
    };
    auto weight_fixed = [&](u32x4 v, const Piece &p, int c0) {
        if (short_w) return v;
        const int left = weight_left(p, c0);
        if (__any(left < 8)) v = left <= 0 ? zero4 : shifted(v, weight_back(left));
        return v;
    };
    auto patch_lds = [&](int buf, int dst) { return reinterpret_cast<u32x4 *>(smem + t.patch_off + buf * t.stage_bytes + dst); };
    auto weight_lds = [&](int buf, int dst) { return reinterpret_cast<u32x4 *>(smem + t.weight_off + buf * t.stage_bytes + dst); };

    // The bias is asked for at once, of a single chunk here, of several behind their loop: a load behind a store is waited for
    // together with the store's acknowledgement (1024 x 1024 x 3 -> 144, 7 x 7 stride 4: a store of 20 300 clocks, 5200 so).  Four channels
    // at a time, in tiles that end past Cout too: by channel their 64 loads and addresses took 3.5 us of 8 x 512 x 198 x 59 -> 96, 1 x 1 stride 2
    // (56.2 -> 52.7).
    const int cl = 4 * (lane >> 5);                       // acc[i][4 g + e] of a lane is channel co0 + 32 i + 8 g + cl + e
    const bool all = co0 + CO <= a.Cout;                  // uniform
    half4v bias[TCO][4];
    auto load_bias = [&]() {
        const half_t *from = a.bias ? a.bias : a.w;       // (Cout halves there too)
        if (all) {
#pragma unroll
            for (int i = 0; i < TCO; i++)
#pragma unroll
                for (int g = 0; g < 4; g++) __builtin_memcpy(&bias[i][g], from + co0 + cl + 32 * i + 8 * g, 8);
        } else if (a.Cout >= 4) {                         // moved back to end inside; `bias_of` shifts
#pragma unroll
            for (int i = 0; i < TCO; i++)
#pragma unroll
                for (int g = 0; g < 4; g++) __builtin_memcpy(&bias[i][g], from + min(co0 + cl + 32 * i + 8 * g, a.Cout - 4), 8);
        } else {
#pragma unroll
            for (int i = 0; i < TCO; i++)
#pragma unroll
                for (int g = 0; g < 4; g++)
#pragma unroll
                    for (int e = 0; e < 4; e++) bias[i][g][e] = i + g == 0 ? from[min(e, a.Cout - 1)] : (half_t)0.0f;
        }
    };
    auto bias_of = [&](int i, int g) {
        const int gone = co0 + 32 * i + 8 * g + cl - (a.Cout - 4);
        if (all || a.Cout < 4) return bias[i][g];
        return __builtin_bit_cast(half4v, __builtin_bit_cast(uint64_t, bias[i][g]) >> (gone > 0 ? 16 * (gone & 3) : 0));      // (past Cout, from four on, nothing is stored)
    };
    if (CHUNKS == 1) load_bias();
    float16v acc[TCO];

    // A single chunk of any size goes to LDS in batches; of several, every thread carries the same few pieces of each.
    Piece pp[PP], wp[WP];
    struct Set { u32x4 p[PP], w[WP]; };
    constexpr bool TWO = TCO <= 2;
    Set set0, set1;
    auto load = [&](Set &v, int ch) {
#pragma unroll
        for (int i = 0; i < WP; i++) v.w[i] = weight_load(wp[i], ch * t.CC);
#pragma unroll
        for (int i = 0; i < PP; i++) v.p[i] = patch_load(pp[i], ch * t.CC);
    };
    // A wave issues a vector instruction every eight clocks at best, so the pieces of a chunk that exists whole take none but
    // their loads: 32-bit offsets from a base that moves in scalar registers, no tests.
    const int nwhole = t.kc % 8 == 0 && !narrow && !short_w ? a.Cin / t.CC : 0;
    auto load_whole = [&](Set &v, int ch) {
        const char *wbase = reinterpret_cast<const char *>(a.w + ch * t.CC * taps), *xbase = reinterpret_cast<const char *>(x + (long)ch * t.CC * HiWi);
#pragma unroll
        for (int i = 0; i < WP; i++) __builtin_memcpy(&v.w[i], wbase + (uint32_t)wp[i].src * 2u, 16);
#pragma unroll
        for (int i = 0; i < PP; i++) __builtin_memcpy(&v.p[i], xbase + (uint32_t)pp[i].src * 2u, 16);
    };
    // Chunk ch goes to LDS.  Pieces outside the image or past kc were zeroed in both stages at the start and stay so.
    auto put = [&](Set &v, int ch) {
        const int buf = ch & 1, c0 = ch * t.CC;
        const bool whole = ch < nwhole;                  // uniform
#pragma unroll
        for (int i = 0; i < WP; i++)
            if (wp[i].have) *weight_lds(buf, wp[i].dst) = whole ? v.w[i] : weight_fixed(v.w[i], wp[i], c0);
#pragma unroll
        for (int i = 0; i < PP; i++)
            if (pp[i].have) {
                if (whole) {
                    if (__any(pp[i].gone)) v.p[i] = shifted(v.p[i], pp[i].gone);
                } else v.p[i] = patch_fixed(v.p[i], pp[i], c0);
                *patch_lds(buf, pp[i].dst) = v.p[i];
            }
    };
    const bool one = CHUNKS == 1 || (CHUNKS == 0 && t.nchunk == 1);
    if (one) {
        // In batches of a few pieces a thread, each one trip to memory.
        const int wend = weight_end(t.kc, CRS, 0), wgone = weight_cut(wend);
        auto stage = [&](auto P_, auto W_) __attribute__((always_inline)) {
            constexpr int P1 = decltype(P_)::value, W1 = decltype(W_)::value;
            for (int d0 = 0, c0 = 0; d0 < t.patch_pieces || c0 < t.weight_pieces; d0 += NT * P1, c0 += NT * W1) {
                Piece pq[P1], wq[W1];
                u32x4 pv[P1], wv[W1];
                if (d0 < t.patch_pieces)                  // uniform, as all four
#pragma unroll
                    for (int i = 0; i < P1; i++) { pq[i] = patch_of(d0 + tid + i * NT); pv[i] = patch_load(pq[i], 0); }
                if (c0 < t.weight_pieces)
#pragma unroll
                    for (int i = 0; i < W1; i++) { wq[i] = weight_of(c0 + tid + i * NT); wv[i] = weight_load(wq[i], 0); }
                if (d0 < t.patch_pieces)
#pragma unroll
                    for (int i = 0; i < P1; i++) {
                        pv[i] = patch_fixed(pv[i], pq[i], 0);
                        if (d0 + tid + i * NT < t.patch_pieces) *patch_lds(0, pq[i].dst) = pv[i];
                    }
                if (c0 < t.weight_pieces)
#pragma unroll
                    for (int i = 0; i < W1; i++) {
                        if (!short_w) {
                            const u32x4 cut = shifted(wv[i], wgone);
                            wv[i] = wq[i].lim + 8 > wend ? cut : wv[i];
                            wv[i] = wq[i].have && wq[i].lim < wend ? wv[i] : zero4;
                        }
                        if (c0 + tid + i * NT < t.weight_pieces) *weight_lds(0, wq[i].dst) = wv[i];
                    }
            }
        };
        using std::integral_constant;
        if (t.patch_pieces <= NT && t.weight_pieces <= 2 * NT) stage(integral_constant<int, 1>{}, integral_constant<int, 2>{});
        else stage(integral_constant<int, 4>{}, integral_constant<int, (TCO > 2 ? 7 : 5)>{});
    } else {
#pragma unroll
        for (int i = 0; i < WP; i++) wp[i] = weight_of(tid + i * NT);
#pragma unroll
        for (int i = 0; i < PP; i++) pp[i] = patch_of(tid + i * NT);
        load(set0, 0);
        if (TWO) load(set1, 1);
        put(set0, 0);
#pragma unroll
        for (int i = 0; i < WP; i++)
            if (!wp[i].have && tid + i * NT < t.weight_pieces) { *weight_lds(0, wp[i].dst) = zero4; *weight_lds(1, wp[i].dst) = zero4; }
#pragma unroll
        for (int i = 0; i < PP; i++)
            if (!pp[i].have && tid + i * NT < t.patch_pieces) { *patch_lds(0, pp[i].dst) = zero4; *patch_lds(1, pp[i].dst) = zero4; }
    }
    if (tid < t.nbuf) *patch_lds(tid, zero_at * 2) = zero4;
    __syncthreads();

#pragma unroll
    for (int i = 0; i < TCO; i++)
#pragma unroll
        for (int r = 0; r < 16; r++) acc[i][r] = 0.0f;

    // this lane's pixel: its origin in the patch
    int lx;
    const int px = pw * 32 + (lane & 31), ly = over(px, t.TW, t.div_tw, lx), h8 = (lane >> 5) * 8;
    const int origin = ly * a.sy * t.PCL + lx * a.sx + (ix0 - xa);
    const int whole = t.kc / 16;                         // steps with sixteen k of the chunk
    auto compute = [&](int buf) {
        const half_t *patch = reinterpret_cast<const half_t *>(smem + t.patch_off + buf * t.stage_bytes), *mine = patch + origin;
        const half_t *wl = reinterpret_cast<const half_t *>(smem + t.weight_off + buf * t.stage_bytes) + (lane & 31) * t.WLD + h8;
        auto gather = [&](const u16x8 off, bool ends) {
            half8v f;
#pragma unroll
            for (int e = 0; e < 8; e++) f[e] = ends && off[e] == zero_at ? patch[zero_at] : mine[off[e]];
            return f;
        };
        auto table = [&](int s) { return *reinterpret_cast<const u16x8 *>(tab + s * 16 + h8); };
        auto products = [&](int s, const half8v fb) {
#pragma unroll
            for (int i = 0; i < TCO; i++)
                acc[i] = __builtin_amdgcn_mfma_f32_32x32x16_f16(*reinterpret_cast<const half8v *>(wl + i * 32 * t.WLD + s * 16), fb, acc[i], 0, 0, 0);
        };
        // Two steps at a time: a step alone is a chain of two LDS trips (table, pixels) behind which its products wait.
        constexpr int U = 2;
        int s = kg;
        for (; s + (U - 1) * KG < whole; s += U * KG) {
            u16x8 off[U];
            half8v fb[U];
#pragma unroll
            for (int u = 0; u < U; u++) off[u] = table(s + u * KG);
#pragma unroll
            for (int u = 0; u < U; u++) fb[u] = gather(off[u], false);
#pragma unroll
            for (int u = 0; u < U; u++) products(s + u * KG, fb[u]);
        }
        for (; s < t.ksteps; s += KG) products(s, gather(table(s), s == whole));
    };
    // Chunk ch is computed while ch + 1 waits in one register set and ch + 2 is on its way into the other: with one set a
    // chunk took a whole trip to memory (2.7 us) whatever its size (and still does with more output channels than registers
    // for two).
    auto turn = [&](Set &now, Set &next, int ch, bool fast) {
        constexpr int AHEAD = TWO ? 2 : 1;
        if (fast) load_whole(now, ch + AHEAD);
        else if (ch + AHEAD < t.nchunk) load(now, ch + AHEAD);
        compute(ch & 1);
        if (ch + 1 < t.nchunk) put(TWO ? next : now, ch + 1);
        __syncthreads();
    };
    int ch = 0;
    if (one) {
        compute(0);
        if constexpr (KG > 1) __syncthreads();            // (below, the groups' sums lie over the operands)
    } else if constexpr (TWO) {
        for (; ch + 3 < nwhole; ch += 2) {
            turn(set0, set1, ch, true);
            turn(set1, set0, ch + 1, true);
        }
        for (; ch < t.nchunk; ch++) {
            const bool fast = ch + 2 < nwhole;
            if (ch & 1) turn(set1, set0, ch, fast);
            else turn(set0, set1, ch, fast);
        }
    } else {
        for (; ch + 1 < nwhole; ch++) turn(set0, set0, ch, true);
        for (; ch < t.nchunk; ch++) turn(set0, set0, ch, false);
    }
    if constexpr (KG > 1) {
        float *part = reinterpret_cast<float *>(smem);      // the operand stages are done with
        if (kg > 0) {
#pragma unroll
            for (int i = 0; i < TCO; i++)
#pragma unroll
                for (int r = 0; r < 16; r++) part[(((kg - 1) * TCO + i) * 16 + r) * (PW * 64) + pw * 64 + lane] = acc[i][r];
        }
        __syncthreads();
        if (kg > 0) return;
        auto add = [&](int i, int g) __attribute__((always_inline)) {
#pragma unroll
            for (int r = 0; r < 16; r++) acc[i][r] += part[((g * TCO + i) * 16 + r) * (PW * 64) + pw * 64 + lane];
        };
        if constexpr (TCO > 2) {
#pragma unroll
            for (int i = 0; i < TCO; i++) {
#pragma unroll
                for (int g = 0; g < KG - 1; g++) add(i, g);
                // left to the stores, behind their conditions, 192 parts waited in scratch memory (8 x 512 x 198 x 59 -> 96: 52.7 -> 41.4 us)
                asm volatile("" : "+v"(acc[i]));
            }
        } else {
#pragma unroll
            for (int g = 0; g < KG - 1; g++)
#pragma unroll
                for (int i = 0; i < TCO; i++) add(i, g);
        }
    }
    if (CHUNKS != 1) load_bias();
    const int oy = oy0 + ly, ox = ox0 + lx;
    const int plane = a.OH * a.OW;                        // Cout planes of an image fit 31 bits
    char *out = reinterpret_cast<char *>(reinterpret_cast<half_t *>(a.out) + (long)blockIdx.z * a.Cout * plane);
    const uint32_t step = (uint32_t)plane * 2u;
    auto rounded = [&](float v0, float v1) {
        half2v v = {(half_t)v0, (half_t)v1};
        if (a.relu) v = __builtin_elementwise_max(v, half2v{(half_t)0.0f, (half_t)0.0f});
        return __builtin_bit_cast(uint32_t, v);
    };
#pragma unroll
    for (int i = 0; i < TCO; i++)
#pragma unroll
        for (int g = 0; g < 4; g++) {
            const half4v b = bias_of(i, g);
#pragma unroll
            for (int e = 0; e < 4; e++) acc[i][4 * g + e] += a.bias ? (float)b[e] : 0.0f;
        }
    // Four lanes, four neighbouring pixels of a row, hold four channels each: they exchange, so that a lane stores four pixels of one
    // channel, eight bytes at any address (by pixel where the row ends between them).
    const int q = lane & 3, left = a.OW - (ox - q);       // pixels of the row from the four's first on
    const bool odd = lane & 1, upper = lane & 2, row_in = oy < a.OH && ly < t.TH && left > 0;
    uint32_t at = (uint32_t)((co0 + cl + q) * plane + oy * a.OW + ox - q) * 2u;
    const bool cut = __any(row_in && left < 4);
#pragma unroll
    for (int i = 0; i < TCO; i++)
#pragma unroll
        for (int g = 0; g < 4; g++, at += 8 * step) {
            // even lanes keep channels 0 and 2 of their own and the next pixel, odd ones 1 and 3 of the one before and their own
            const uint32_t p01 = rounded(acc[i][4 * g], acc[i][4 * g + 1]), p23 = rounded(acc[i][4 * g + 2], acc[i][4 * g + 3]);
            const uint32_t n01 = __builtin_amdgcn_update_dpp(0, p01, 0xB1, 0xF, 0xF, true), n23 = __builtin_amdgcn_update_dpp(0, p23, 0xB1, 0xF, 0xF, true);
            const uint32_t a01 = odd ? pack_hi(n01, p01) : pack_lo(p01, n01), a23 = odd ? pack_hi(n23, p23) : pack_lo(p23, n23);
            const uint32_t give = upper ? a01 : a23, keep = upper ? a23 : a01, got = __builtin_amdgcn_update_dpp(0, give, 0x4E, 0xF, 0xF, true);
            const u32x2 v = {upper ? got : keep, upper ? keep : got};
            if (row_in && (all || co0 + 32 * i + 8 * g + cl + q < a.Cout)) {
                if (left >= 4) __builtin_memcpy(out + at, &v, 8);
                else if (cut) {
                    const half4v h = __builtin_bit_cast(half4v, v);
#pragma unroll
                    for (int e = 0; e < 3; e++) if (e < left) *reinterpret_cast<half_t *>(out + at + 2 * e) = h[e];
                }
            }
        }
}

template <int PW, int KG, int TCO>
int launch(const TileConv &t, hipStream_t st) {
    constexpr int parts = (KG - 1) * TCO * 16 * PW * 64 * 4;
    const int lds = (int)std::max<int64_t>(t.patch_off + (int64_t)t.nbuf * t.stage_bytes, parts);
    const dim3 grid((unsigned)(t.tiles_x * t.tiles_y), (unsigned)ceil_div(t.a.Cout, 32 * TCO), (unsigned)t.a.N);
    if (t.a.Wi < 8 || weights_by_element(t.kc, t.a.Cin * t.a.KH * t.a.KW)) hipLaunchKernelGGL((conv_tile_kernel<PW, KG, TCO, 0>), grid, dim3(PW * KG * 64), lds, st, t);
    else if (t.nchunk == 1) hipLaunchKernelGGL((conv_tile_kernel<PW, KG, TCO, 1>), grid, dim3(PW * KG * 64), lds, st, t);
    else hipLaunchKernelGGL((conv_tile_kernel<PW, KG, TCO, 2>), grid, dim3(PW * KG * 64), lds, st, t);
    return hipGetLastError() == hipSuccess ? MI_OK : MI_ERROR_LAUNCH;
}

template <typename F>
int with_shape(const Shape &s, F f) {
#define ONE(P, K, T) if (s.pw == P && s.kg == K && s.tco == T) return f(std::integral_constant<int, P>{}, std::integral_constant<int, K>{}, std::integral_constant<int, T>{});
    ONE(8, 1, 1) ONE(8, 1, 2) ONE(8, 1, 3) ONE(8, 1, 4) ONE(8, 1, 5) ONE(4, 1, 1) ONE(4, 1, 2) ONE(4, 1, 3) ONE(4, 1, 5) ONE(4, 2, 1) ONE(4, 2, 2) ONE(4, 2, 3) ONE(4, 2, 4) ONE(2, 4, 1) ONE(2, 4, 2) ONE(2, 4, 4) ONE(2, 2, 1) ONE(2, 2, 2)
#undef ONE
    return MI_DECLINE_EXTENT;
}

// The last choices of this thread: an estimate of every shape takes the host a few microseconds.
struct Choice { int cus; ConvShape key; double us; Shape s; TilePlan t; };
const Choice &choice_of(const ConvArgs &a) {
    static thread_local Choice table[16] = {};
    const int cus = mi_num_cus();
    Choice &e = table[shape_hash(a, cus) >> 28];
    if (e.cus != cus || !same_shape(e.key, a)) {
        e.cus = cus;
        e.key = a;
        if (!choose(a, cus, e.t, e.s, e.us)) e.us = 1e30;
    }
    return e;
}

}  // namespace

double mi_conv_tile_us(const ConvArgs &a) { return choice_of(a).us; }

int mi_conv_tile(const ConvArgs &a, hipStream_t st) {
    const Choice &e = choice_of(a);
    if (e.us >= 1e30) return MI_DECLINE_EXTENT;
    const TileConv t{e.t, a, recip_of(e.t.tiles_x), recip_of(a.KH * a.KW), recip_of(a.KW), recip_of(e.t.TW), recip_of(e.t.PC8), recip_of(e.t.PR), recip_of(e.t.wpieces)};
    return with_shape(e.s, [&](auto P, auto K, auto T) { return launch<P, K, T>(t, st); });
}

int mi_conv_tile_init() {
    int bad = 0;
    for (const Shape &s : SHAPES)
        bad |= with_shape(s, [&](auto P, auto K, auto T) {
            auto up = [](auto kern) { return hipFuncSetAttribute(reinterpret_cast<const void *>(kern), hipFuncAttributeMaxDynamicSharedMemorySize, LDS_MAX) == hipSuccess ? 0 : 1; };
            return up(conv_tile_kernel<P, K, T, 0>) | up(conv_tile_kernel<P, K, T, 1>) | up(conv_tile_kernel<P, K, T, 2>);
        });
    return bad;
}
