// Fused attention for gfx950 on 32-query workgroups: grids that the 128- and 256-query forms of sdpa.hip leave the chip
// idle on, and head sizes that those pad to 64 or 96.
#include "sdpa_common.hpp"

namespace {

// A workgroup owns 32 queries of one (head, batch); its NW waves take the 32-key tiles w, w + NW, ... of the keys, each with its
// own softmax state and its own stretch of LDS, and share nothing until the (O, M, l) of all waves meet in LDS at the end
// (the rescaling identity of flash.jl:1385-1391).  No barrier in the loop, nothing staged for anyone else.
//
// What bounds it is the vector ALU and the latency of a tile's serial chain (first product, exponentials, second product),
// so what counts is waves: everything a wave holds fits 128 registers at head size 64 and 8.5 KB of LDS, four waves a SIMD.
// To that end K and V travel global -> LDS without passing through registers (global_load_lds_dwordx4), into one buffer
// each: the next tile's K is requested when this tile's fragments have been read, the next V likewise, so a request has
// the other product and the exponentials to arrive under.  (Fragments straight from memory -- a lane per key row -- cost
// the CU's vector-memory path a cache line per 32 bytes.)  A second buffer a wave, query tiles that start at different
// keys, and 64 queries a wave measured the same or slower (6 heads x 1370: 12.3 us; 13.8, 13.4 and 14.7).
//
// A direct load cannot pad, so the EC 16-byte chunks of a row (EC = E / 8) are permuted instead: K row r holds chunk c at
// c ^ kswz(r) such that any eight rows' reads of one chunk fall into eight bank groups, V row r at c ^ vswz(r) such that the
// four rows of a transposing read do.  Rows of nine chunks (72) need none for K.
//
// Products, register layouts and the lazily moved reference point M are flash_fwd_kernel's: S^T = K Q^T, O^T = V^T P^T, -M in
// the first product's accumulators.
//
// KEYS, DENSE: what a mask is.  KEYS: fp16 and of the key alone, copied to LDS once; it joins in one more k-step as (mask, mask) x
// (log2(e) split into two positive fp16 parts), so that -inf stays -inf.  DENSE (with F32): anything else -- any strides, addresses
// and either type -- read a tile ahead, a lane the sixteen values of its query, and added to the scores in fp32.  The loads are the
// compiler's, whose waits know nothing of the requests: they are waited for where K has had a tile's time to land, before V is
// asked for.  Such calls went to a workgroup per query row: 5 x 12 x 3559 x 3559 x 16 11 170 us, 6 x 20 x 189 x 189 x 16 88 -> 8.6,
// 14 x 12 x 53 x 53 x 64 22 -> 6.9, 4 x 4 x 77 x 3238 57 -> 22, 4 x 6 x 257 x 257 35 -> 9.7.
//
// F32: calls of few queries, which the rows kernel answers with its scores and probabilities in fp32.  Nothing is rounded to fp16
// here either: Q goes into the product as it lies and the scale joins the scores in fp32 (with the mask, times log2(e), from
// an fp32 row), a probability enters the second product as two fp16 values (hi, lo) that hold 22 bits of 2^10 p, and what a
// product adds up is kept short -- 16 head dims, 32 keys -- and joined with vector adds, whose roundings are smaller than the
// matrix unit's.  Relative error against 64 bits (2-norm, random operands, fp32 result; rows kernel | here | fp16 operands):
// 23 x 300 x 64: 1.48e-7 | 1.45e-7 | 2.7e-4; 63 x 4000 x 64: 2.4e-7 | 2.0e-7 | 3.0e-4; 23 x 300 x 128: 1.66e-7 | 1.58e-7.  Only at head size
// 72 it is larger, 1.57e-7 | 1.65e-7: there fp32 results stay with the rows kernel (fp16 ones are off by their rounding, 2.1e-4,
// either way).
// EARLY: a tile's V is read from LDS ahead of its exponentials, into registers that the others fill behind them, so that the wait for
// the reads is none.  A wave needs 16 registers more at head size 64 and 24 at 72.  us, late | early: 6 heads x 1370 x 64 11.9 | 11.6, 12 x 4 x
// 504 x 16 6.95 | 6.7, 2 x 16 x 5 x 3966 x 32 with padding 21.7 | 20.1 (with Q's wait out of the loop), 20 heads x 290 x 64 5.54 | 5.46.  Where the
// registers cost a wave that the grid has, it is late: 16 x 3644 x 285 x 64 12.6 | 14.7, 5 x 20 x 1085 x 72 79 | 80.  Dense masks take
// the registers for theirs: 16 x 4 x 77 x 128 6.2 | 6.6.
// Waves a SIMD that the registers of an instance are budgeted for.
enum TileMask { NO_MASK, KEYS, DENSE };
constexpr bool tile_early(int EC, bool F32, int MASK) { return MASK != DENSE && (F32 || EC != 9); }
constexpr int tile_waves(int EC, bool F32, int MASK, bool EARLY) { return EC == 8 && !F32 && EARLY ? 3 : EC == 16 ? 2 : EC == 9 ? (F32 ? 2 : 3) : EC == 8 && F32 ? (MASK == DENSE ? 2 : 3) : MASK == DENSE ? 3 : 4; }

template <int EC, int NW, int MASK, bool F32, bool EARLY = tile_early(EC, F32, MASK)>
__global__ __launch_bounds__(NW * 64, tile_waves(EC, F32, MASK, EARLY)) void flash_tile_kernel(SdpaArgs p) {
    typedef std::conditional_t<F32, float, half_t> mask_t;
    static_assert(MASK != DENSE || F32, "calls with fp16 probabilities and such a mask run flash_fwd_kernel");
    constexpr int E = EC * 8, KS = (E + 15) / 16, ET = (E + 31) / 32;
    constexpr int TILE_BYTES = 32 * EC * 16, NI = (32 * EC + 63) / 64;      // one operand's tile; 1 KB requests for it
    constexpr int WPART = (ET * 16 + 2) * 256, WSTRIDE = WPART > 2 * TILE_BYTES ? WPART : 2 * TILE_BYTES;
    constexpr float UP = F32 ? 1024.0f : 1.0f, TH = F32 ? 4.0f : 8.0f;      // probabilities times UP stay in fp16 range
    extern __shared__ __align__(16) char smem[];
    stage_tile_args(p);
    const int lane = threadIdx.x & 63, wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
    const int hl = lane >> 5, l32 = lane & 31;
    char *const wave_lds = smem + wave * WSTRIDE;
    const uint32_t lds0 = (uint32_t)(uintptr_t)(__attribute__((address_space(3))) char *)smem + wave * WSTRIDE;
    mask_t *const Ms = reinterpret_cast<mask_t *>(smem + NW * WSTRIDE);

    // workgroups are dealt to the 8 XCDs round robin: each gets a contiguous run, so a head's query tiles share an L2
    int qblk, h, b;
    {
        const int total = p.nqb * p.H * p.B, xcd = blockIdx.x & 7, full = total >> 3, rem = total & 7;
        unsigned x, y;
        const unsigned hb = divide(xcd * full + min(xcd, rem) + (blockIdx.x >> 3), p.nqb, p.div_x, x);
        // (said to be scalar: the carry of a quotient was kept in a vector register as far as the mask copy, which spilled)
        b = __builtin_amdgcn_readfirstlane(divide(hb, p.H, p.div_h, y));
        qblk = __builtin_amdgcn_readfirstlane(x);
        h = __builtin_amdgcn_readfirstlane(y);
    }
    const int q0 = qblk * 32;
    const half_t *qb = p.q + h * p.qs[2] + b * p.qs[3];
    int Lk = p.Lk;
    if (p.kv_len) Lk = max(0, min(Lk, p.kv_len[b]));
    const int nt = (Lk + 31) / 32, last = Lk - 1;             // rows past the end re-read the last key that counts: whatever lies behind it, a weight of zero would not hide an infinity
    const float c = p.scale * LOG2E;

    u32x4 qraw[KS];
    {
        const int qr = min(q0 + l32, p.Lq - 1);
#pragma unroll
        for (int ks = 0; ks < KS; ks++) {
            const u32x4 z = {0u, 0u, 0u, 0u};
            const int e = 16 * ks + 8 * hl;
            qraw[ks] = e < E ? ldg16(qb + (long)qr * p.qs[1] + e) : z;
        }
    }
    auto kswz = [](int r) { return EC == 9 ? 0 : EC == 2 ? (r >> 2) & 1 : EC == 4 ? (r >> 1) & 3 : r & 7; };
    auto vswz = [](int r) { return EC == 8 || EC == 16 ? (r & 3) * 2 : 0; };
    // Requests: lane and request i stand for 16-byte slot s = 64 i + lane of the tile, row s / EC, position s % EC.
    const char *const kbase = reinterpret_cast<const char *>(p.k + h * p.ks[2] + b * p.ks[3]);
    const char *const vbase = reinterpret_cast<const char *>(p.v + h * p.vs[2] + b * p.vs[3]);
    const uint32_t kpitch = (uint32_t)p.ks[1] * 2, vpitch = (uint32_t)p.vs[1] * 2;
    uint32_t koff[NI], voff[NI];
#pragma unroll
    for (int i = 0; i < NI; i++) {
        const int s = 64 * i + lane, row = s / EC, pos = s % EC;
        koff[i] = row * kpitch + (pos ^ kswz(row)) * 16;
        voff[i] = row * vpitch + (pos ^ vswz(row)) * 16;
    }
    auto request = [&](bool is_k, int tile) {
        const char *org = (is_k ? kbase : vbase) + (long)tile * 32 * (is_k ? kpitch : vpitch);
        const int over = tile * 32 + 31 - last;                   // rows of the tile past the last key
        const uint32_t dst = lds0 + (is_k ? 0 : TILE_BYTES);
        if (over <= 0) {                                          // uniform
            if constexpr ((32 * EC) % 64 == 0) {
                asm volatile("s_mov_b32 m0, %0" ::"s"(dst) : "memory");
#pragma unroll
                for (int i = 0; i < NI; i++)
                    asm volatile("s_nop 0\n\tglobal_load_lds_dwordx4 %0, %1\n\ts_add_u32 m0, m0, 0x400" ::"v"(is_k ? koff[i] : voff[i]), "s"(org) : "memory", "scc");
                return;
            }
        }
#pragma unroll
        for (int i = 0; i < NI; i++) {
            const int s = 64 * i + lane;
            uint32_t off = is_k ? koff[i] : voff[i];
            if (over > 0) off -= max(0, s / EC - (31 - over)) * (is_k ? kpitch : vpitch);
            if ((32 * EC) % 64 == 0 || s < 32 * EC)
                asm volatile("s_mov_b32 m0, %2\n\ts_nop 0\n\tglobal_load_lds_dwordx4 %0, %1" ::"v"(off), "s"(org), "s"(F32 ? __builtin_amdgcn_readfirstlane(dst + i * 1024) : dst + i * 1024) : "memory");
        }
    };
    if (wave < nt) { request(true, wave); request(false, wave); }
    if constexpr (MASK == KEYS) {
        const unsigned short *mrow = reinterpret_cast<const unsigned short *>(p.bias) + (long)h * p.bs[2] + (long)b * p.bs[3];
        for (int i = threadIdx.x; i < nt * 32; i += NW * 64) {
            const half_t m = __builtin_bit_cast(half_t, i < p.Lk ? mrow[(long)i * p.bs[0]] : (unsigned short)0);
            if constexpr (F32) Ms[i] = (float)m * LOG2E;
            else Ms[i] = m;
        }
    }
    half8v qf[KS];
#pragma unroll
    for (int ks = 0; ks < KS; ks++) {
        const half8v t = as_half8(qraw[ks]);
#pragma unroll
        for (int j = 0; j < 8; j++) qf[ks][j] = F32 ? t[j] : (half_t)((float)t[j] * c);
    }
    // (F32 does nothing to Q that would wait for it: left to its first use, in the loop, that wait is one for the next K in every turn)
    if constexpr (F32 && MASK != DENSE) {
#pragma unroll
        for (int ks = 0; ks < KS; ks++) {
            u32x4 w = __builtin_bit_cast(u32x4, qf[ks]);
            asm volatile("" : "+v"(w));
            qf[ks] = __builtin_bit_cast(half8v, w);
        }
    }
    float16v o_acc[ET], negm;
#pragma unroll
    for (int r = 0; r < 16; r++) negm[r] = 0.0f;
#pragma unroll
    for (int t = 0; t < ET; t++) o_acc[t] = negm;
    float m_run = F32 ? 0.0f : -INFINITY, l_run = 0.0f;           // no reference point yet: negm is 0
    half8v qext;
    if constexpr (MASK == KEYS) {
#pragma unroll
        for (int j = 0; j < 8; j++) qext[j] = (half_t)0.0f;
        if (hl == 0) { qext[0] = (half_t)1.4423828125f; qext[1] = (half_t)(1.44269504088896340736f - 1.4423828125f); }
        __syncthreads();                                          // the mask row is in place
    }
    const int vk = (lane & 15) >> 2;                              // key of a transposing read's four
    auto vchunk = [&](int t) { return min(4 * t + 2 * ((lane >> 4) & 1) + ((lane & 3) >> 1), EC - 1) ^ vswz(vk); };
    auto probs = [&](const float16v &sx, half8v (&pf)[2], half8v (&lo)[2], float &l) {
#pragma unroll
        for (int r = 0; r < 16; r += 2) {
            const float p0 = __builtin_amdgcn_exp2f(sx[r]) * UP, p1 = __builtin_amdgcn_exp2f(sx[r + 1]) * UP;
            pf[r >> 3][r & 7] = (half_t)p0;
            pf[r >> 3][(r & 7) + 1] = (half_t)p1;
            if constexpr (F32) {
                lo[r >> 3][r & 7] = (half_t)(p0 - (float)(half_t)p0);
                lo[r >> 3][(r & 7) + 1] = (half_t)(p1 - (float)(half_t)p1);
            }
            l += p0 + p1;
        }
    };
    // DENSE: the lane's sixteen values of a tile, keys 32 tile + 8 g + 4 hl .. +3, raw as they lie in memory (g holds four values:
    // four words of fp32, two of fp16).  A tile that the keys end in, and keys apart in memory, are read by element, past the end
    // the last one again: such keys' scores are cut.
    u32x4 mraw[MASK == DENSE ? 4 : 1];
    const char *drow = nullptr;
    if constexpr (MASK == DENSE) drow = reinterpret_cast<const char *>(p.bias) + ((long)min(q0 + l32, p.Lq - 1) * p.bs[1] + (long)h * p.bs[2] + (long)b * p.bs[3]) * (p.bias_f32 ? 4 : 2);
    auto mask_load = [&](int tile) {
        const bool run = p.bs[0] == 1 && tile * 32 + 32 <= p.Lk;          // uniform
        if (p.bias_f32) {
#pragma unroll
            for (int g = 0; g < 4; g++) {
                const int key = tile * 32 + 8 * g + 4 * hl;
                if (run) __builtin_memcpy(&mraw[g], drow + (long)key * 4, 16);
                else {
#pragma unroll
                    for (int e = 0; e < 4; e++) mraw[g][e] = reinterpret_cast<const uint32_t *>(drow)[(long)min(key + e, p.Lk - 1) * p.bs[0]];
                }
            }
        } else {
#pragma unroll
            for (int g = 0; g < 4; g++) {
                const int key = tile * 32 + 8 * g + 4 * hl;
                if (run) {
                    u32x2 t;
                    __builtin_memcpy(&t, drow + (long)key * 2, 8);      // at any address
                    mraw[g][0] = t[0]; mraw[g][1] = t[1];
                } else {
                    unsigned short t[4];
#pragma unroll
                    for (int e = 0; e < 4; e++) t[e] = reinterpret_cast<const unsigned short *>(drow)[(long)min(key + e, p.Lk - 1) * p.bs[0]];
                    mraw[g][0] = t[0] | (uint32_t)t[1] << 16; mraw[g][1] = t[2] | (uint32_t)t[3] << 16;
                }
            }
        }
    };
    float16v ms;                                                  // KEYS: times log2(e); DENSE: as it came
    auto mask_take = [&]() {
        if (p.bias_f32) {
#pragma unroll
            for (int r = 0; r < 16; r++) { const uint32_t w = mraw[r >> 2][r & 3]; ms[r] = __builtin_bit_cast(float, w); }
        } else {
#pragma unroll
            for (int r = 0; r < 16; r += 2) {
                const uint32_t w = mraw[r >> 2][(r & 3) >> 1];
                const half2v t = __builtin_bit_cast(half2v, w);
                ms[r] = (float)t[0]; ms[r + 1] = (float)t[1];
            }
        }
#pragma unroll
        for (int r = 0; r < 16; r++) asm volatile("" : "+v"(ms[r]));      // here, not where they are used
    };
    if constexpr (MASK == DENSE) { if (wave < nt) { mask_load(wave); mask_take(); } }
    bool first = true;
    // Keys that a finite mask excludes (finfo.min: -94 498 here) do not settle M, which scores formed against it would pay with
    // their last bits: see flash_fwd_kernel's FLOOR.
    constexpr float FLOOR = MASK && !F32 ? -1024.0f : -INFINITY;      // (F32: the scores are kept, and scaled again)
    const char *const kt_lds = wave_lds, *const vt_lds = wave_lds + TILE_BYTES;
    for (int tile = wave; tile < nt; tile += NW) {
        const bool more = tile + NW < nt;
        asm volatile("s_waitcnt vmcnt(%0)" ::"n"(NI) : "memory");          // K has landed; V may be on its way
        half8v kf[KS];
#pragma unroll
        for (int ks = 0; ks < KS; ks++)
            kf[ks] = *reinterpret_cast<const half8v *>(kt_lds + (l32 * EC + (min(2 * ks + hl, EC - 1) ^ kswz(l32))) * 16);
        half8v kx = {};
        if constexpr (MASK == KEYS && F32) {
#pragma unroll
            for (int g = 0; g < 4; g++) {
                const float4v m = *reinterpret_cast<const float4v *>(Ms + tile * 32 + 8 * g + 4 * hl);
#pragma unroll
                for (int e = 0; e < 4; e++) ms[4 * g + e] = m[e];
            }
        } else if constexpr (MASK == KEYS) {
            const half_t m = Ms[tile * 32 + l32];
            kx[0] = hl == 0 ? m : (half_t)0.0f;
            kx[1] = kx[0];
        }
        asm volatile("s_waitcnt lgkmcnt(0)" ::: "memory");
        if (more) {
            request(true, tile + NW);
            if constexpr (MASK == DENSE) mask_load(tile + NW);
        }
        float16v sc = __builtin_amdgcn_mfma_f32_32x32x16_f16(kf[0], qf[0], negm, 0, 0, 0);
#pragma unroll
        for (int ks = 1; ks < KS; ks++) {
            if constexpr (F32) {
                const float16v part = __builtin_amdgcn_mfma_f32_32x32x16_f16(kf[ks], qf[ks], negm, 0, 0, 0);      // (negm stays 0)
#pragma unroll
                for (int r = 0; r < 16; r++) sc[r] += part[r];
            } else sc = __builtin_amdgcn_mfma_f32_32x32x16_f16(kf[ks], qf[ks], sc, 0, 0, 0);
        }
        if constexpr (MASK == KEYS && !F32) sc = __builtin_amdgcn_mfma_f32_32x32x16_f16(kx, qext, sc, 0, 0, 0);
        auto cut = [&]() {                                        // the ragged last tile: excluded keys get -inf
            if (tile * 32 + 32 > Lk) {
#pragma unroll
                for (int r = 0; r < 16; r++)
                    if (tile * 32 + 8 * (r >> 2) + 4 * hl + (r & 3) >= Lk) sc[r] = -INFINITY;
            }
        };
        // DENSE: score and mask are rounded into one number, once, and M is the largest such number itself.  However large a mask
        // (1e9 swallows its score, finfo.min times log2(e) would be infinite), no score of M's tile is above M, and a row of
        // equal numbers is a row of equal weights.  (Error with fp32 results against the row kernel's, over 80 calls of 16 to 128 wide
        // heads, 60 to 1500 keys and scores of standard deviation 1 and 3: 3.5 % less on average, at 64 2 % more.  One log2(e) inside the
        // fma instead of behind the difference, where M is small enough for it, took off 0.3 % more and cost 3 % of the time.)
        if constexpr (MASK == DENSE) {
#pragma unroll
            for (int r = 0; r < 16; r++) sc[r] = fmaf(sc[r], p.scale, ms[r]);
            cut();
        }
        const float16v raw = sc;
        auto scale = [&]() {
            if constexpr (MASK == DENSE) {
#pragma unroll
                for (int r = 0; r < 16; r++) sc[r] = (raw[r] - m_run) * LOG2E;
                return;
            }
#pragma unroll
            for (int r = 0; r < 16; r++) sc[r] = fmaf(raw[r], c, MASK ? ms[r] - m_run : -m_run);
            cut();
        };
        if constexpr (F32) scale();
        else cut();
        half8v vf[ET][2];
        auto read_v = [&]() __attribute__((always_inline)) {
            if (more) asm volatile("s_waitcnt vmcnt(%0)" ::"n"(NI) : "memory");        // V has landed; the next K may be on its way
            else asm volatile("s_waitcnt vmcnt(0)" ::: "memory");
#pragma unroll
            for (int t = 0; t < ET; t++)
#pragma unroll
                for (int bb = 0; bb < 2; bb++) {
                    const char *vq = vt_lds + ((16 * bb + 4 * hl + vk) * EC + vchunk(t)) * 16 + (lane & 1) * 8;
                    const short4v lo = __builtin_amdgcn_ds_read_tr16_b64_v4i16((__attribute__((address_space(3))) short4v *)vq);
                    const short4v hi = __builtin_amdgcn_ds_read_tr16_b64_v4i16((__attribute__((address_space(3))) short4v *)(vq + 8 * EC * 16));
                    const short8v both = {lo[0], lo[1], lo[2], lo[3], hi[0], hi[1], hi[2], hi[3]};
                    vf[t][bb] = __builtin_bit_cast(half8v, both);
                }
        };
        if constexpr (EARLY) read_v();                            // comes back under the exponentials
        half8v pf[2], lo[2];
        float l_new = l_run;
        probs(sc, pf, lo, l_new);
        if (__any(first || !(l_new - l_run < 65504.0f))) {        // flash_fwd_kernel says why
            const float16v &from = MASK == DENSE ? raw : sc;
            float tmax = fmaxf(from[0], from[1]);
#pragma unroll
            for (int r = 2; r < 16; r += 2) tmax = fmaxf(fmaxf(tmax, from[r]), from[r + 1]);
            const float top = fmaxf(tmax, __shfl_xor(tmax, 32, 64)), mx = MASK == DENSE ? (top - m_run) * LOG2E : top;
            const bool grow = (mx > TH || first) && top > FLOOR;
            float d = grow ? mx : 0.0f, alpha = first ? 0.0f : __builtin_amdgcn_exp2f(-d);
            float to = MASK == DENSE ? (grow ? top : m_run) : first ? d : m_run + d;
            if constexpr (!F32) {
#pragma unroll
                for (int r = 0; r < 16; r++) negm[r] = -to;
            }
            if constexpr (MASK && !F32) {
                if (first && !grow) {                             // masked keys only, so far
                    to = fmaxf(m_run, mx);
                    d = to == -INFINITY ? 0.0f : to;
                    alpha = to == -INFINITY ? 0.0f : __builtin_amdgcn_exp2f(m_run - to);
                }
            }
            m_run = to;
            l_run *= alpha;
            if constexpr (F32) scale();
            else {
#pragma unroll
                for (int r = 0; r < 16; r++) sc[r] -= d;
            }
#pragma unroll
            for (int t = 0; t < ET; t++)
#pragma unroll
                for (int r = 0; r < 16; r++) o_acc[t][r] *= alpha;
            l_new = l_run;
            probs(sc, pf, lo, l_new);
            first = first && !grow;                               // the reference point is found with the first key that counts
        }
        l_run = l_new;
        if constexpr (MASK == DENSE) { if (more) mask_take(); }
        if constexpr (!EARLY) read_v();
        asm volatile("s_waitcnt lgkmcnt(0)" ::: "memory");
        if (more) request(false, tile + NW);
#pragma unroll
        for (int t = 0; t < ET; t++) {
            if constexpr (F32) {                                  // the small parts first
                float16v part = __builtin_amdgcn_mfma_f32_32x32x16_f16(vf[t][0], lo[0], negm, 0, 0, 0);
                part = __builtin_amdgcn_mfma_f32_32x32x16_f16(vf[t][1], lo[1], part, 0, 0, 0);
                part = __builtin_amdgcn_mfma_f32_32x32x16_f16(vf[t][0], pf[0], part, 0, 0, 0);
                part = __builtin_amdgcn_mfma_f32_32x32x16_f16(vf[t][1], pf[1], part, 0, 0, 0);
#pragma unroll
                for (int r = 0; r < 16; r++) o_acc[t][r] += part[r];
            } else {
#pragma unroll
                for (int bb = 0; bb < 2; bb++) o_acc[t] = __builtin_amdgcn_mfma_f32_32x32x16_f16(vf[t][bb], pf[bb], o_acc[t], 0, 0, 0);
            }
        }
    }
    // The waves' partials, lane-major, each into its own stretch, then every wave finishes (t, g) pairs: head dims
    // 32 t + 8 g + 4 hl .. +3 of its lane's query.
    float *xo = reinterpret_cast<float *>(wave_lds);
#pragma unroll
    for (int t = 0; t < ET; t++)
#pragma unroll
        for (int r4 = 0; r4 < 4; r4++) {
            const float4v v = {o_acc[t][4 * r4], o_acc[t][4 * r4 + 1], o_acc[t][4 * r4 + 2], o_acc[t][4 * r4 + 3]};
            *reinterpret_cast<float4v *>(xo + (t * 4 + r4) * 256 + lane * 4) = v;
        }
    xo[ET * 1024 + lane] = m_run;
    xo[ET * 1024 + 64 + lane] = l_run + __shfl_xor(l_run, 32, 64);      // both lanes of a query hold half of its row sum
    __syncthreads();
    float aw[NW], mm = -INFINITY, den = 0.0f;
#pragma unroll
    for (int w = 0; w < NW; w++) {
        const float *xw = reinterpret_cast<const float *>(smem + w * WSTRIDE) + ET * 1024;
        aw[w] = xw[64 + lane] > 0.0f ? xw[lane] : -INFINITY;  // a wave that saw no valid key has a meaningless reference point
        mm = fmaxf(mm, aw[w]);
    }
#pragma unroll
    for (int w = 0; w < NW; w++) {
        const float *xw = reinterpret_cast<const float *>(smem + w * WSTRIDE) + ET * 1024;
        aw[w] = aw[w] == -INFINITY ? 0.0f : __builtin_amdgcn_exp2f(MASK == DENSE ? (aw[w] - mm) * LOG2E : aw[w] - mm);
        den += aw[w] * xw[64 + lane];
    }
    const float inv = den > 0.0f ? 1.0f / den : 0.0f;
    const int qi = q0 + l32;
    for (int tg = wave; tg < EC; tg += NW) {
        float4v o = {0.0f, 0.0f, 0.0f, 0.0f};
#pragma unroll
        for (int w = 0; w < NW; w++) {
            const float4v x = *reinterpret_cast<const float4v *>(reinterpret_cast<const float *>(smem + w * WSTRIDE) + tg * 256 + lane * 4);
#pragma unroll
            for (int i = 0; i < 4; i++) o[i] += aw[w] * x[i];
        }
        if (qi < p.Lq) {
            const long off = (long)b * p.os[3] + (long)h * p.os[2] + (long)qi * p.os[1] + 8 * tg + 4 * hl;
            if (p.out_f32) {
                const float4v r = {o[0] * inv, o[1] * inv, o[2] * inv, o[3] * inv};
                *reinterpret_cast<float4v *>(reinterpret_cast<float *>(p.out) + off) = r;
            } else {
                const half4v r = {(half_t)(o[0] * inv), (half_t)(o[1] * inv), (half_t)(o[2] * inv), (half_t)(o[3] * inv)};
                *reinterpret_cast<half4v *>(reinterpret_cast<half_t *>(p.out) + off) = r;
            }
        }
    }
}

template <int EC, int NW>
constexpr int tile_lds_bytes() {
    constexpr int part = ((EC * 8 + 31) / 32 * 16 + 2) * 256, tiles = 2 * 32 * EC * 16;
    return NW * (part > tiles ? part : tiles);
}
template <int EC, int NW, int MASK, bool F32, bool EARLY>
int launch_instance(const SdpaArgs &p, int lds, hipStream_t st) {
    hipLaunchKernelGGL((flash_tile_kernel<EC, NW, MASK, F32, EARLY>), dim3((unsigned)(p.nqb * p.H * p.B)), dim3(NW * 64), lds, st, p);
    return hipGetLastError() == hipSuccess ? MI_OK : MI_ERROR_LAUNCH;
}
template <int EC, int NW, int MASK, bool F32>
int launch_tiles(const SdpaArgs &p, int lds, hipStream_t st) {
    constexpr bool early = tile_early(EC, F32, MASK);
    if constexpr (early && tile_waves(EC, F32, MASK, true) < tile_waves(EC, F32, MASK, false)) {
        // as long as all waves of the grid find room at once (four SIMDs a CU)
        if ((int64_t)p.nqb * p.H * p.B * NW > (int64_t)4 * tile_waves(EC, F32, MASK, true) * mi_num_cus()) return launch_instance<EC, NW, MASK, F32, false>(p, lds, st);
    }
    return launch_instance<EC, NW, MASK, F32, early>(p, lds, st);
}
template <int EC, int NW, bool F32>
int launch_tiles(const SdpaArgs &p, TileMask mask, hipStream_t st) {
    const int lds = tile_lds_bytes<EC, NW>();
    if (mask == KEYS) return launch_tiles<EC, NW, KEYS, F32>(p, lds + (int)ceil_div(p.Lk, 32) * 32 * (F32 ? 4 : 2), st);
    if (mask == DENSE) {
        if constexpr (F32) return launch_tiles<EC, NW, DENSE, true>(p, lds, st);
        else return MI_DECLINE_BIAS;
    }
    return launch_tiles<EC, NW, NO_MASK, F32>(p, lds, st);
}
template <int EC, bool F32>
int launch_waves(const SdpaArgs &p, int waves, TileMask mask, hipStream_t st) {
    return waves == 2 ? launch_tiles<EC, 2, F32>(p, mask, st) : waves == 4 ? launch_tiles<EC, 4, F32>(p, mask, st) : launch_tiles<EC, 8, F32>(p, mask, st);
}
template <int EC, int NW, int MASK, bool F32>
int raise_one(int lds) {
    int bad = 0;
    if constexpr (tile_early(EC, F32, MASK))
        bad |= hipFuncSetAttribute(reinterpret_cast<const void *>(flash_tile_kernel<EC, NW, MASK, F32, true>), hipFuncAttributeMaxDynamicSharedMemorySize, lds) != hipSuccess;
    if constexpr (!tile_early(EC, F32, MASK) || tile_waves(EC, F32, MASK, true) < tile_waves(EC, F32, MASK, false))
        bad |= hipFuncSetAttribute(reinterpret_cast<const void *>(flash_tile_kernel<EC, NW, MASK, F32, false>), hipFuncAttributeMaxDynamicSharedMemorySize, lds) != hipSuccess;
    return bad;
}
template <int EC, int NW, bool F32>
int raise() {
    const int lds = tile_lds_bytes<EC, NW>();
    return raise_one<EC, NW, KEYS, F32>(lds + (F32 ? 4 : 2) * MI_SDPA_TILE_KEYMASK_MAX) | raise_one<EC, NW, DENSE, true>(lds) | raise_one<EC, NW, NO_MASK, F32>(lds);
}
template <int EC>
int raise_all() { return raise<EC, 2, false>() | raise<EC, 4, false>() | raise<EC, 8, false>() | raise<EC, 2, true>() | raise<EC, 4, true>() | raise<EC, 8, true>(); }

}  // namespace

// Head sizes: those of this package's models and tests.  The chunk permutations hold for rows of 2, 4, 8, 9 and 16 chunks; 40, 48, 80,
// 96 and the rest run the padded forms of flash_fwd_kernel, which no figure here has been taken against.
bool mi_sdpa_tile_head_size(int64_t E) { return E == 16 || E == 32 || E == 64 || E == 72 || E == 128; }
// An fp16 mask of the key alone whose row fits the LDS is copied there; one that differs from query to query is read where it lies.  (An
// fp32 one of the key alone keeps the rows kernel, the fused one its own blocks.)
bool mi_sdpa_tile_keymask(const SdpaArgs &p) { return p.bias && !p.bias_f32 && (p.bs[1] == 0 || p.Lq == 1) && p.Lk <= MI_SDPA_TILE_KEYMASK_MAX; }
bool mi_sdpa_tile_takes(const SdpaArgs &p) {
    if (!mi_sdpa_tile_head_size(p.E)) return false;
    if (p.bias && !mi_sdpa_tile_keymask(p) && p.bs[1] == 0) return false;
    // a launch has fewer than 2^32 threads along its one dimension (grids of this size run two waves a workgroup)
    if ((int64_t)ceil_div(p.Lq, 32) * p.H * p.B * 128 > UINT32_MAX) return false;
    // per-lane load offsets are 32-bit byte offsets from a tile's first row
    return p.ks[1] >= 0 && p.vs[1] >= 0 && p.ks[1] * 64 < (1l << 31) && p.vs[1] * 64 < (1l << 31);
}

int mi_sdpa_tile_launch(const SdpaArgs &args, int waves, bool f32, hipStream_t st) {
    if (!mi_sdpa_tile_takes(args)) return MI_DECLINE_EXTENT;
    SdpaArgs p = args;
    p.nqb = (int)ceil_div(p.Lq, 32);
    p.div_x = recip_of(p.nqb);
    const TileMask mask = !p.bias ? NO_MASK : mi_sdpa_tile_keymask(p) ? KEYS : DENSE;
    switch (p.E) {
    case 16: return f32 ? launch_waves<2, true>(p, waves, mask, st) : launch_waves<2, false>(p, waves, mask, st);
    case 32: return f32 ? launch_waves<4, true>(p, waves, mask, st) : launch_waves<4, false>(p, waves, mask, st);
    case 64: return f32 ? launch_waves<8, true>(p, waves, mask, st) : launch_waves<8, false>(p, waves, mask, st);
    case 72: return f32 ? launch_waves<9, true>(p, waves, mask, st) : launch_waves<9, false>(p, waves, mask, st);
    default: return f32 ? launch_waves<16, true>(p, waves, mask, st) : launch_waves<16, false>(p, waves, mask, st);
    }
}

int mi_sdpa_tile_init() {
    return raise_all<2>() | raise_all<4>() | raise_all<8>() | raise_all<9>() | raise_all<16>();
}
