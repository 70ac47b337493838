// Attention of a single query row per (head, batch), a decode step's, for gfx950: one launch, the new key and value written to
// the cache on the way where the caller asks for it.
#include "sdpa_common.hpp"
#include <algorithm>
#include <atomic>

namespace {

// Arrival counters and partials of the split form: a launch takes the next of SD_BANKS banks, so launches in flight
// together on one GPU (up to SD_BANKS of them) do not touch each other's.  Zero when the module loads; every launch
// leaves its counters at zero.
constexpr int SD_BANKS = 16, SD_TICKETS = 4096, SD_PART_FLOATS = 1 << 16;
static __device__ unsigned sd_ticket_words[SD_BANKS * SD_TICKETS];
static __device__ __align__(256) float sd_part_words[SD_BANKS * SD_PART_FLOATS];
constexpr int SD_MAX_DEVICES = 64;
unsigned *g_sd_tickets[SD_MAX_DEVICES] = {};
float *g_sd_parts[SD_MAX_DEVICES] = {};
std::atomic<unsigned> g_sd_launch{0};

// Single query row per (head, batch): 8-wave workgroups, `nsplit` of them per row, each over its share of the key
// range.  A wave takes keys 8 at a time (8 lanes per key, one 16-byte chunk of the head dim each) with a stride of
// 64 keys, in rounds of U passes whose K and V loads are all issued before the first is used; up to eight passes are one round,
// MANY: more are taken in rounds of four, the next round's requested before the current round is consumed (64 registers of them, so that two
// workgroups fit on a CU: 20 x 32 heads over 1500 keys 36.9 us, in rounds of five 39.6, of six 40.0).
//
// Such a launch moves a few MB, so its duration is a chain of trips to memory.  Every address is therefore made
// independent of loaded data: the key range is cut by the cache's capacity (p.Lk), not by kv_len, and keys are
// requested up to the capacity -- valid memory whatever the length -- together with the length itself, the query
// and the new row; the length only masks scores afterwards.  No load stands behind a condition of its lane's: where the two sides
// meet the compiler waits for it and for all before it.  Head dims below 64 repeat their last chunk, with a query of zeros.
//
// A round's scores come first, then one maximum for the whole wave (of its eight groups of lanes), then the probabilities: nothing in
// a round waits for another key's exponential, and the groups' sums meet without rescaling.
//
// nsplit > 1: the workgroups of one row run on one XCD (workgroup ids are dealt to XCDs round robin, so ids that
// differ by multiples of 8 share an L2), write their partial (max, sum, o[E]) to part_o / part_ml, and take a ticket;
// whoever draws the last ticket merges the partials in split order -- so the result does not depend on who that
// is -- writes the row and puts the ticket counter back to zero.  Nobody waits for anybody: every workgroup exits
// after its own work.  The exchange stays inside that one L2 and one wave: a partial is written with plain stores, waited for
// (vmcnt) and followed by the ticket, an atomic the L2 performs; the merging wave reads with loads that go to
// the L2.  A device-scope release per workgroup instead (__threadfence) writes the whole L2 back each time: measured
// 63 us for 320 workgroups against 6 us unsplit.  The host only splits on a device whose probe showed the round-robin
// placement this relies on.
constexpr int SD_U_MANY = 4;
template <int U, bool MANY, bool APPEND, bool FAR = false>
__global__ __launch_bounds__(512) void sdpa_decode_kernel(SdpaArgs p) {
    __shared__ float red_ml[8][2];
    __shared__ float red_o[8][64];
    stage_decode_args(p);
    const int tid = threadIdx.x, lane = tid & 63, wave = __builtin_amdgcn_readfirstlane(tid >> 6);
    const int grp = lane >> 3, cl = lane & 7;
    const int S = p.nsplit;
    const int xcd = blockIdx.x & 7, slot = blockIdx.x >> 3;
    unsigned split_, h_;
    const int unit = __builtin_amdgcn_readfirstlane((int)divide(slot, S, p.div_split, split_) * 8 + xcd), split = __builtin_amdgcn_readfirstlane((int)split_);
    if (unit >= p.H * p.B) return;                       // the grid is padded to whole groups of 8 rows
    const unsigned b = __builtin_amdgcn_readfirstlane(divide(unit, p.H, p.div_h, h_)), h = __builtin_amdgcn_readfirstlane(h_);
    const int cap = p.Lk;
    const int npass = (cap + 63) >> 6, per = p.per;
    const int t_lo = split * per, t_hi = min(npass, t_lo + per);
    half_t *kb = const_cast<half_t *>(p.k) + h * p.ks[2] + b * p.ks[3];
    half_t *vb = const_cast<half_t *>(p.v) + h * p.vs[2] + b * p.vs[3];
    const bool eok = cl * 8 < p.E;
    const int e0 = min(cl * 8, p.E - 8);
    const int n_read = *(p.kv_len ? p.kv_len + b : reinterpret_cast<const int *>(p.q));
    const int first = 8 * wave;                          // pass t of this wave covers keys 64 t + first + grp
    struct Round { u32x4 k[U], v[U]; };
    // Byte offsets in a head's keys and values are 32 bits, so that the clamp at the capacity is one of offsets (FAR: any strides).
    const unsigned kstride = (unsigned)p.ks[1] * 2, vstride = (unsigned)p.vs[1] * 2;
    const unsigned k_lane = (first + grp) * kstride + 2 * e0, v_lane = (first + grp) * vstride + 2 * e0;
    const unsigned k_last = (cap - 1) * kstride + 2 * e0, v_last = (cap - 1) * vstride + 2 * e0;
    auto at = [](const half_t *base, unsigned bytes) { return ldg16(reinterpret_cast<const half_t *>(reinterpret_cast<const char *>(base) + bytes)); };
    auto fetch = [&](Round &r, int t0) {
#pragma unroll
        for (int u = 0; u < U; u++) {
            // (passes past the end read the last one again, keys past the capacity the last key)
            const int k0 = 64 * min(t0 + u, t_hi - 1);
            if constexpr (FAR) {
                const long key = min(k0 + first + grp, cap - 1);
                r.k[u] = ldg16(kb + key * p.ks[1] + e0);
                r.v[u] = ldg16(vb + key * p.vs[1] + e0);
            } else {
                r.k[u] = at(kb, min(k0 * kstride + k_lane, k_last));
                r.v[u] = at(vb, min(k0 * vstride + v_lane, v_last));
            }
        }
    };
    const u32x4 qraw = ldg16(p.q + h * p.qs[2] + b * p.qs[3] + e0);
    u32x4 kn, vn;                                        // the row that this step appends
    if constexpr (APPEND) {
        kn = ldg16(p.k_new + h * p.ns[2] + b * p.ns[3] + e0);
        vn = ldg16(p.v_new + h * p.ns[2] + b * p.ns[3] + e0);
    }
    Round cur, nxt;
    fetch(cur, t_lo);
    if constexpr (MANY) fetch(nxt, t_lo + U);
    __builtin_amdgcn_sched_barrier(0);                   // nothing above waits
    float qv[8];
    {
        const half8v t = as_half8(qraw);
        const float scale = eok ? p.scale * LOG2E : 0.0f;
#pragma unroll
        for (int j = 0; j < 8; j++) qv[j] = (float)t[j] * scale;
    }
    // a length past the capacity: the cache is full, the new row is neither stored nor attended
    const int n_raw = p.kv_len ? __builtin_amdgcn_readfirstlane(n_read) : cap;
    const int Lk = max(0, min(cap, n_raw));
    const int fresh = APPEND && n_raw <= cap ? Lk - 1 : -1;
    float m = -INFINITY, l = 0.0f, acc[8];
#pragma unroll
    for (int j = 0; j < 8; j++) acc[j] = 0.0f;
    auto consume = [&](Round &r, int t0) {
        float sc[U];
        float top = -INFINITY;
#pragma unroll
        for (int u = 0; u < U; u++) {
            const int k0 = 64 * (t0 + u) + first, key = k0 + grp;
            sc[u] = -INFINITY;
            if (t0 + u < t_hi && k0 < Lk) {              // uniform
                if (APPEND && fresh >= k0 && fresh < k0 + 8) {      // uniform; exactly eight lanes of one workgroup own it
                    const bool mine = key == fresh;
                    r.k[u] = mine ? kn : r.k[u];
                    r.v[u] = mine ? vn : r.v[u];
                    if (mine && eok) {
                        *reinterpret_cast<u32x4 *>(kb + (long)key * p.ks[1] + e0) = kn;
                        *reinterpret_cast<u32x4 *>(vb + (long)key * p.vs[1] + e0) = vn;
                    }
                }
                const half8v kt = as_half8(r.k[u]);
                float d = 0.0f, d4 = 0.0f;                   // (two chains: a shorter one rounds less)
#pragma unroll
                for (int j = 0; j < 4; j++) { d = fmaf(qv[j], (float)kt[j], d); d4 = fmaf(qv[j + 4], (float)kt[j + 4], d4); }
                d = eok ? d + d4 : 0.0f;
                d += lane_xor<1>(d);
                d += lane_xor<2>(d);
                d += lane_xor<4>(d);
                sc[u] = key < Lk ? d : -INFINITY;
                top = fmaxf(top, sc[u]);
            }
        }
        {   // over the wave's groups of eight lanes
            float x = top, y = top;
            swap_rows32(x, y); top = fmaxf(x, y);
            x = top; y = top;
            swap_rows16(x, y); top = fmaxf(x, y);
            top = fmaxf(top, lane_xor<8>(top));
        }
        const float mn = fmaxf(m, top), mu = mn == -INFINITY ? 0.0f : mn;
        if constexpr (MANY) {
            const float al = __builtin_amdgcn_exp2f(m - mu);
            l *= al;
#pragma unroll
            for (int j = 0; j < 8; j++) acc[j] *= al;
        }
        m = mn;
#pragma unroll
        for (int u = 0; u < U; u++) {
            const int k0 = 64 * (t0 + u) + first;
            if (t0 + u < t_hi && k0 < Lk) {
                const float pw = __builtin_amdgcn_exp2f(sc[u] - mu);
                l += pw;
                u32x4 vr = r.v[u];
                const u32x4 z = {0u, 0u, 0u, 0u};
                if (k0 + 8 > Lk) vr = k0 + grp < Lk ? vr : z;      // a weight of zero would not hide what an unwritten slot may hold
                const half8v vt = as_half8(vr);
#pragma unroll
                for (int j = 0; j < 8; j++) acc[j] = fmaf(pw, (float)vt[j], acc[j]);
            }
        }
    };
    if constexpr (!MANY) consume(cur, t_lo);
    else {
        for (int t0 = t_lo;; t0 += 2 * U) {
            consume(cur, t0);
            if (t0 + 2 * U >= t_hi) { consume(nxt, t0 + U); break; }
            fetch(cur, t0 + 2 * U);
            consume(nxt, t0 + U);
            if (t0 + 3 * U >= t_hi) { consume(cur, t0 + 2 * U); break; }
            fetch(nxt, t0 + 3 * U);
        }
    }
    // The sums of the wave's eight groups, each exchange halving what a lane still holds: lane (h, r, i, cl) of the bits 5, 4, 3 and 2..0
    // ends with element 8 cl + 4 h + 2 r + i.
#pragma unroll
    for (int j = 0; j < 4; j++) { swap_rows32(acc[j], acc[j + 4]); acc[j] += acc[j + 4]; }
#pragma unroll
    for (int j = 0; j < 2; j++) { swap_rows16(acc[j], acc[j + 2]); acc[j] += acc[j + 2]; }
    const bool odd = lane & 8;
    const float o = (odd ? acc[1] : acc[0]) + lane_xor<8>(odd ? acc[0] : acc[1]);
    {
        float x = l, y = l;
        swap_rows32(x, y); l = x + y;
        x = l; y = l;
        swap_rows16(x, y); l = x + y;
        l += lane_xor<8>(l);
    }
    red_o[wave][8 * cl + ((lane >> 5) & 1) * 4 + ((lane >> 4) & 1) * 2 + ((lane >> 3) & 1)] = o;
    if (lane == 0) { red_ml[wave][0] = m; red_ml[wave][1] = l; }
    __syncthreads();
    if (wave > 0) return;                                // what is left is one wave's
    float mm = -INFINITY, L = 0.0f, O = 0.0f;
#pragma unroll
    for (int w = 0; w < 8; w++) mm = fmaxf(mm, red_ml[w][0]);
    {
        const float mu = mm == -INFINITY ? 0.0f : mm;
#pragma unroll
        for (int w = 0; w < 8; w++) {
            const float a = __builtin_amdgcn_exp2f(red_ml[w][0] - mu);
            L += a * red_ml[w][1];
            O += a * red_o[w][lane];
        }
    }
    if (S > 1) {                                         // uniform
        const long row = (long)unit * S + split;
        if (lane < p.E) p.part_o[row * p.E + lane] = O;
        if (lane == 0) { p.part_ml[row * 2] = mm; p.part_ml[row * 2 + 1] = L; }
        asm volatile("s_waitcnt vmcnt(0)" ::: "memory");  // the partial has reached the L2 before the ticket is drawn
        unsigned t = 0;
        if (lane == 0) t = __hip_atomic_fetch_add(p.tickets + unit, 1u, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
        if (__builtin_amdgcn_readfirstlane(t) != (unsigned)(S - 1)) return;
        if (lane == 0) __hip_atomic_store(p.tickets + unit, 0u, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);   // ready for the next launch
        mm = -INFINITY; L = 0.0f; O = 0.0f;
        const long r0 = (long)unit * S;
        const int el = min(lane, p.E - 1);
        for (int s0 = 0; s0 < S; s0 += 8) {
            float ms[8], ls[8], os_[8];
#pragma unroll
            for (int j = 0; j < 8; j++) {
                const long r = r0 + min(s0 + j, S - 1);
                // read at the L2, past this compute unit's own cache
                ms[j] = __hip_atomic_load(p.part_ml + r * 2, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
                ls[j] = __hip_atomic_load(p.part_ml + r * 2 + 1, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
                os_[j] = __hip_atomic_load(p.part_o + r * p.E + el, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
            }
            float mb = mm;
#pragma unroll
            for (int j = 0; j < 8; j++) {
                if (s0 + j >= S) ms[j] = -INFINITY;      // a split past the end: weight 0
                mb = fmaxf(mb, ms[j]);
            }
            const float mu = mb == -INFINITY ? 0.0f : mb;
            const float a0 = __builtin_amdgcn_exp2f(mm - mu);
            L *= a0; O *= a0;
#pragma unroll
            for (int j = 0; j < 8; j++) {
                const float a = __builtin_amdgcn_exp2f(ms[j] - mu);
                L += a * ls[j];
                O += a * os_[j];
            }
            mm = mb;
        }
    }
    if (lane < p.E) {
        const float r = L > 0.0f ? O / L : 0.0f;
        const long oo = (long)b * p.os[3] + (long)h * p.os[2] + (long)lane * p.os[0];
        if (p.out_f32) reinterpret_cast<float *>(p.out)[oo] = r;
        else reinterpret_cast<half_t *>(p.out)[oo] = (half_t)r;
    }
}

}  // namespace

// Head dim <= 64, no additive mask; the rest goes to sdpa_rows_kernel (+ sdpa_merge_kernel).
bool mi_sdpa_decode_takes(const SdpaArgs &a) {
    return a.Lq == 1 && !a.bias && a.E <= 64 && a.Lk >= 1 && (int64_t)a.H * a.B <= SD_TICKETS;
}

// Twenty heads alone leave most of the chip idle and give each workgroup a long chain of keys, so a long key range is cut over several
// workgroups per row, at most one per compute unit.
int mi_sdpa_decode_splits(int64_t E, int64_t Lk, int64_t H, int64_t B) {
    const int64_t units = H * B, passes = ceil_div(Lk, 64);
    // The exchange adds about 1.5 us of its own (partial out, ticket, partials in: three trips in a row), a pass 0.3: 448 keys stay whole
    // (20 heads, keys in the L2 and from memory: 4.6 and 5.2 us, cut in two 5.3 and 5.7), 1500 are cut four ways
    // (eight rows of passes in three splits 6.2 and 7.9 against 5.9 and 7.3, three in eight 6.2 and 7.0).
    int64_t want = mi_num_cus() / units;                 // at most one workgroup per compute unit
    if (want > ceil_div(passes, 6)) want = ceil_div(passes, 6);
    if (passes <= 8) want = 1;
    if (want > 32) want = 32;
    while (want > 1 && units * want * (E + 2) > SD_PART_FLOATS) want--;
    if (want < 1) want = 1;
    // no empty split: with `per` passes each, the last one must still start inside the range
    while (want > 1 && ceil_div(passes, want) * (want - 1) >= passes) want--;
    return (int)want;
}

// Fills in the split count and, for a split launch, this launch's bank of counters and partials, and launches.
int mi_sdpa_decode_launch(const SdpaArgs &args, hipStream_t st) {
    SdpaArgs a = args;
    a.nsplit = mi_sdpa_decode_splits(a.E, a.Lk, a.H, a.B);
    if (a.nsplit > 1) {
        int dev = -1;
        if (!mi_xcd_round_robin() || hipGetDevice(&dev) != hipSuccess || dev < 0 || dev >= SD_MAX_DEVICES || !g_sd_tickets[dev]) a.nsplit = 1;
        else {
            const unsigned bank = g_sd_launch++ % SD_BANKS;
            a.tickets = g_sd_tickets[dev] + (size_t)bank * SD_TICKETS;
            a.part_o = g_sd_parts[dev] + (size_t)bank * SD_PART_FLOATS;
            a.part_ml = a.part_o + (size_t)a.H * a.B * a.nsplit * a.E;
        }
    }
    a.per = (int)ceil_div(ceil_div(a.Lk, 64), a.nsplit);
    a.div_split = recip_of(a.nsplit);
    const dim3 grid((unsigned)ceil_div((int64_t)a.H * a.B, 8) * 8 * a.nsplit);
    // byte offsets beyond 32 bits, those of passes past the end included (a single key has none)
    if (a.Lk > 1 && (a.ks[1] < 0 || a.vs[1] < 0 || (int64_t)(a.Lk + 64) * std::max(a.ks[1], a.vs[1]) * 2 >= (1ll << 32))) {
        if (a.k_new) hipLaunchKernelGGL((sdpa_decode_kernel<SD_U_MANY, true, true, true>), grid, dim3(512), 0, st, a);
        else         hipLaunchKernelGGL((sdpa_decode_kernel<SD_U_MANY, true, false, true>), grid, dim3(512), 0, st, a);
        return hipGetLastError() == hipSuccess ? MI_OK : MI_ERROR_LAUNCH;
    }
    auto go = [&](auto U, auto MANY) {
        if (a.k_new) hipLaunchKernelGGL((sdpa_decode_kernel<decltype(U)::value, decltype(MANY)::value, true>), grid, dim3(512), 0, st, a);
        else         hipLaunchKernelGGL((sdpa_decode_kernel<decltype(U)::value, decltype(MANY)::value, false>), grid, dim3(512), 0, st, a);
    };
    using std::integral_constant;
    switch (a.per) {                                     // one round of exactly as many passes as there are, up to eight
        case 1: go(integral_constant<int, 1>{}, std::false_type{}); break;
        case 2: go(integral_constant<int, 2>{}, std::false_type{}); break;
        case 3: go(integral_constant<int, 3>{}, std::false_type{}); break;
        case 4: go(integral_constant<int, 4>{}, std::false_type{}); break;
        case 5: go(integral_constant<int, 5>{}, std::false_type{}); break;
        case 6: go(integral_constant<int, 6>{}, std::false_type{}); break;
        case 7: go(integral_constant<int, 7>{}, std::false_type{}); break;
        case 8: go(integral_constant<int, 8>{}, std::false_type{}); break;
        default: go(integral_constant<int, SD_U_MANY>{}, std::true_type{});
    }
    return hipGetLastError() == hipSuccess ? MI_OK : MI_ERROR_LAUNCH;
}

// This device's copies of the counters and partials (zeroed at load; never named in host code again).
void mi_sdpa_decode_init() {
    int dev = -1;
    void *t = nullptr, *pw = nullptr;
    if (hipGetDevice(&dev) == hipSuccess && dev >= 0 && dev < SD_MAX_DEVICES &&
        hipGetSymbolAddress(&t, HIP_SYMBOL(sd_ticket_words)) == hipSuccess && hipGetSymbolAddress(&pw, HIP_SYMBOL(sd_part_words)) == hipSuccess) {
        g_sd_tickets[dev] = reinterpret_cast<unsigned *>(t);
        g_sd_parts[dev] = reinterpret_cast<float *>(pw);
    }
}
