// fp16 GEMM for gfx950: MFMA 32x32x16 f16 with fp32 accumulation, LDS
// double-buffered operand tiles, 128-bit global loads, fused bias / activation /
// residual store.  The four-wave kernel, the plans and the C ABI are here; gemm_skinny.hip has the decode-sized kernels, gemm_pipe.hip has the small tiles, gemm_ring.hip those of small deep grids and the gathered ones of a
// convolution, gemm_any.hip what none of them can address.
//
// Internal problem statement (row-major):  Y[M x N] = A[M x K] . B  (+ bias)
//   A is K-contiguous.  B is either N-contiguous [K][N] (B_KN) or K-contiguous
//   [N][K].  For a linear layer M = tokens, N = features, A = X, B = W.
#include "gemm_common.hpp"
#include "conv_common.hpp"
#include "sk_exchange.hpp"
#include <algorithm>
#include <atomic>

// Arrival flags of the split-K peer reduction (gemm_w4_kernel, SK): SK_BANKS banks of SK_FLAGS words, and as many
// counters behind them (word i's counter is word i + SK_WORDS).  A launch uses the bank its epoch selects, so launches
// that overlap on one GPU (up to SK_BANKS of them) do not see each other's.  Every word is zero when the module loads
// and zero again when a launch ends: the last consumer of a flag clears it (and its counter), so a captured launch --
// whose epoch and bank are fixed at capture -- starts every replay from clean flags.
constexpr int SK_BANKS = 16, SK_FLAGS = 4096, SK_WORDS = SK_BANKS * SK_FLAGS;
static __device__ unsigned sk_flag_words[2 * SK_WORDS];

// Sticky device status word (mi_device_status): kernels OR a bit of enum mi_device_status_bits into word 0 when a
// bounded wait inside a launch gave up; nothing on the device ever clears it.
static __device__ unsigned device_status_words[4];

// Static device scratch of the allocation-free entry point (see mi_gemm_f16_noalloc).
static __device__ __align__(256) unsigned char scratch[MI_NOALLOC_SCRATCH_BYTES];

namespace {

// ------------------------------------------------------------------------------------------
// Split-K without fp32 planes and without a second launch: the two workgroups of a tile (gemm_w4_kernel, SK) exchange
// their partial tiles inside the launch.
//
// Workgroup pid runs on XCD pid % 8 (workgroups are dealt to the XCDs round robin; mi_init checks that this device
// does so and the path stays off otherwise): pid = (slot * 2 + s) * 8 + xcd computes K-slice s of tile xcd * tpx + slot,
// so the partners of a tile share an XCD, i.e. one L2, and are dispatched together.  After its K loop every wave owns
// half of its 64 x 64 accumulators -- the 32-row block s -- writes the other half into its partner's slot of sk_part
// (plain stores: they stay in the shared L2), waits for them to be acknowledged, and raises its flag; it then waits
// (bounded) for the same wave of its partner, adds what it sent in slice order (the result does not depend on which
// workgroup sums), and stores its share through the usual epilogue.  Both workgroups publish before they wait, so the
// waits are not circular among resident workgroups; the launcher only checks that the grid fits an IDLE device in
// one round.  Under overlap (another stream's kernel holding CUs) a partner may not be resident yet: the wait is
// bounded, and a wave that runs into the bound -- or finds its partner on another XCD -- raises the device's sticky
// status word (mi_device_status), stores NaN over its share of Y and releases nothing (sk_exchange.hpp has the
// protocol; tests/sk_exchange_host_test.cpp runs it on CPU threads, with one and with three partners).
// (Four slices of a 128 x 256 tile were built and measured as well: three partners to wait for, 23 MB exchanged at
// 1500 x 5120 -> 1280, 40.8 us against 29.8 us for two slices of 128 x 128.)
struct SkDeviceMem {
    __device__ static unsigned load(const unsigned *p) { return __hip_atomic_load(p, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT); }
    __device__ static void store(unsigned *p, unsigned v) { __hip_atomic_store(p, v, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT); }
    __device__ static unsigned fetch_add(unsigned *p, unsigned v) { return __hip_atomic_fetch_add(p, v, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT); }
    __device__ static void pause() { __builtin_amdgcn_s_sleep(1); }
};
using SkExchange = sk::Exchange<SkDeviceMem>;

// A wave whose exchange failed marks its share of the output instead of storing a plausible sum: NaN in the output
// type over rows [r0, r0 + 32) x columns [c0, c0 + ncols) of the tile.
// (Scalars by value: a reference to the kernel's argument block would force the block into private memory.)
__device__ __noinline__ void sk_poison_region(void *Y, long ldY, int M, int N, int out_f32, int r0, int c0, int ncols, int lane) {
    for (int e = lane; e < 32 * ncols; e += 64) {
        const int m = r0 + e / ncols, n = c0 + e % ncols;
        if (m < M && n < N) {
            const long off = (long)m * ldY + n;
            if (out_f32) reinterpret_cast<unsigned *>(Y)[off] = 0x7fc00000u;
            else reinterpret_cast<unsigned short *>(Y)[off] = (unsigned short)0x7e00u;
        }
    }
}

// The end of a split-K launch whose two K-slices exchange their partial tiles: every wave sends the 32-row block it
// does not keep to its partner, raises its flag, waits (bounded) for the same wave of the partner, sums what arrived
// in slice order and stores its block.
// sk_part[tile][owner][source][wave of NWAVES][column half][4][64 lanes][4]; flags [tile][slice][8].
template <int TM, int TN, int WTM, int WTN, int NWAVES, int LDS_BYTES>
__device__ __forceinline__ void sk_finish(const GemmArgs &p, float16v (&acc)[TN][TM], const half4v (&cb)[TN][4], char *smem, int sk_tile, int sk_s,
                                          int m0, int n0, int wm, int wn, int wave, int lane, long bz) {
    static_assert(TM == 2 && TN == 2, "a wave's 64 x 64 accumulators: two 32-row blocks of two 32 x 32 sub-tiles");
    // four registers per lane and access, 1 KB per wave instruction
    auto part_of = [&](int owner, int src) { return p.sk_part + ((((long)sk_tile * 2 + owner) * 2 + src) * NWAVES + wave) * 2048L + lane * 4; };
    float16v own[2];
    static_for<2>([&](auto J) {
        constexpr int j = decltype(J)::value;
        if (j == sk_s) {                                       // uniform: the block this wave keeps
            own[0] = acc[0][j]; own[1] = acc[1][j];
        } else {
            float *dst = part_of(j, sk_s);
#pragma unroll
            for (int i = 0; i < 2; i++)
#pragma unroll
                for (int r4 = 0; r4 < 4; r4++) {
                    const float4v v = {acc[i][j][4 * r4], acc[i][j][4 * r4 + 1], acc[i][j][4 * r4 + 2], acc[i][j][4 * r4 + 3]};
                    *reinterpret_cast<float4v *>(dst + i * 1024 + r4 * 256) = v;
                }
        }
    });
    // the partials must have reached L2 before the flag can be seen
    asm volatile("s_waitcnt vmcnt(0)" ::: "memory");
    const unsigned my_xcc = __builtin_amdgcn_s_getreg((3 << 11) | 20) & 15u;      // HW_REG_XCC_ID, bits 3:0
    unsigned *myflag = p.sk_flags + ((long)sk_tile * 2 + sk_s) * 8 + wave;
    unsigned *theirs = p.sk_flags + ((long)sk_tile * 2 + (1 - sk_s)) * 8 + wave;
    if (lane == 0) SkExchange::publish(myflag, p.sk_epoch ^ p.sk_pub_xor, my_xcc);
    // Co-residency of the partner is NOT guaranteed (another stream's kernel can hold an XCD's CUs): the bound is the
    // guard, and a wave that runs into it says so.
    const unsigned *const cfl[3] = {theirs, theirs, theirs};
    const sk::WaitResult wr = SkExchange::wait(cfl, 1, p.sk_epoch, my_xcc ^ p.sk_xcc_xor, p.sk_spin);
    asm volatile("" ::: "memory");
    if (wr != sk::ARRIVED) {
        // Loud failure: the sticky status word, NaN over this wave's share of Y, flags left as they are (the host
        // zeroes the banks when it reads the status).  The wave still leaves the kernel normally.
        if (lane == 0) __hip_atomic_fetch_or(p.status, wr == sk::TIMED_OUT ? (unsigned)MI_DEVSTAT_EXCHANGE_TIMEOUT : (unsigned)MI_DEVSTAT_EXCHANGE_XCD,
                                             __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
        // (the exchange runs unbatched launches only: bz = 0)
        sk_poison_region(p.Y, p.ldY, p.M, p.N, p.out_f32, m0 + wm * WTM + 32 * sk_s, n0 + wn * WTN, WTN, lane);
        return;
    }
    // Ordinary loads: this CU has not touched these lines since the kernel began (its L1 was invalidated then), so
    // they come from the L2 the partner's acknowledged stores are in (the wait has checked that it is this XCD's).
    const float *from = part_of(sk_s, 1 - sk_s);
    float4v blk[2][4];
#pragma unroll
    for (int i = 0; i < 2; i++)
#pragma unroll
        for (int r4 = 0; r4 < 4; r4++) blk[i][r4] = *reinterpret_cast<const float4v *>(from + i * 1024 + r4 * 256);
    float16v two[2][1];                                        // summed in slice order, whoever does the summing
#pragma unroll
    for (int i = 0; i < 2; i++)
#pragma unroll
        for (int r = 0; r < 16; r++) two[i][0][r] = sk_s == 0 ? own[i][r] + blk[i][r >> 2][r & 3] : blk[i][r >> 2][r & 3] + own[i][r];
    // What the partner sent has arrived (the sums above used it): this wave clears the partner's flag, so the next
    // launch on this bank, which for a replayed graph carries this same epoch, starts from zero.
    if (lane == 0) SkExchange::release(theirs, theirs + SK_WORDS, 1);
    store_tile<1, 2, WTM, WTN, NWAVES, LDS_BYTES>(p, two, cb, smem, m0 + 32 * sk_s, n0, wm, wn, wave, lane, bz);
}

// ------------------------------------------------------------------------------------------
// Four matrix waves, one per SIMD, each with a BM x BN/4 strip of the tile, and a loader wave.
//
// The ping-pong kernel's 128 x 256 tile spends a third of its K loop in waits: per 64-deep tile its eight 64 x 64
// waves read 8 x 16 KB of fragments for 1024 clocks of MFMAs per SIMD, a SIMD takes 32 B/clock from the LDS, and the
// two phases of a tile came to 1590 clocks (measured with clock stamps; no different with every workgroup on one
// L2-resident tile, so it is not memory).  A wave that owns 128 x 64 reads 24 KB for twice the MFMAs.  With one matrix
// wave per SIMD there is no partner to alternate phases with; instead each wave overlaps its own work: three sets
// of fragment registers (4 A + 2 B fragments of a 16-deep step), the reads of step s + 2 dealt one or two at a time
// between the eight MFMAs of step s -- issued in one burst they held the wave at the LDS queue while its matrix pipe
// ran dry -- and an MFMA in flight does not hold up the wave's LDS instructions.  128 accumulator registers + 72 of
// fragments fit because at most two waves (a matrix wave and the loader) share a SIMD: 256 registers each.
// Measured: 1290 to 1390 clocks a tile, and 1500 x 1280 -> 5120 in 23.1 us against 25.5 to 26.1 us.
//
// One workgroup barrier per tile, B_kt, taken by the matrix waves in the middle of tile kt's third step -- after the
// last fragment read of the tile has returned, before the first read of tile kt + 1 -- and by the loader after it has
// waited for tile kt + 1 to land.  Past B_kt stage kt % 3 is free, and the loader requests tile kt + 3 into it.
template <int BM, int BN, int BK, bool B_KN>
struct DirectTile {
    static constexpr int CPR = BK / 8, ROWB = BK * 2, A_BYTES = BM * ROWB, B_BYTES = BN * ROWB, STAGE_BYTES = A_BYTES + B_BYTES;
    static constexpr int SLOTS_A = A_BYTES / 1024, SLOTS_B = B_BYTES / 1024;      // 1 KB = one wave-wide request
    __device__ __forceinline__ static int rowswz(int r) { return BK == 64 ? (r & 7) ^ ((r >> 3) & 1) : (r >> 2) & 3; }
    // per-lane byte offset, from the tile's origin in memory, of what lands in 1 KB slot s of the A / B part of a stage
    __device__ __forceinline__ static uint32_t a_offset(const GemmArgs &p, int m0, int s, int lane) {
        const int q = s * 64 + lane, r = q / CPR, pos = q % CPR;
        return (uint32_t)(((long)(min(m0 + r, p.M - 1) - m0) * p.ldA + (pos ^ rowswz(r)) * 8) * 2);
    }
    __device__ __forceinline__ static uint32_t b_offset(const GemmArgs &p, int n0, int s, int lane) {
        const int q = s * 64 + lane;
        if (!B_KN) {
            const int r = q / CPR, pos = q % CPR;
            return (uint32_t)(((long)(min(n0 + r, p.N - 1) - n0) * p.ldB + (pos ^ rowswz(r)) * 8) * 2);
        } else {
            constexpr int CPRB = BN / 8;
            const int k = q / CPRB, pos = q % CPRB, j = pos ^ ((k & 3) << 2);
            return (uint32_t)(((long)k * p.ldB + (min(n0 + j * 8, p.NB - 8) - n0)) * 2);
        }
    }
    __device__ __forceinline__ static void request(const char *base, uint32_t off, uint32_t lds_dst) {
        const uint32_t dst = __builtin_amdgcn_readfirstlane(lds_dst);
        asm volatile("s_mov_b32 m0, %2\n\ts_nop 0\n\tglobal_load_lds_dwordx4 %0, %1" ::"v"(off), "s"(base), "s"(dst) : "memory");
    }
};

template <int BM, int BN, int WAVES_M, int WAVES_N, bool B_KN, bool SK = false>
__global__ __launch_bounds__(512) void gemm_w4_kernel(GemmArgs p) {
    constexpr int BK = 64, STAGES = 3, KS = 4;
    using T = DirectTile<BM, BN, BK, B_KN>;
    constexpr int ROWB = T::ROWB, A_BYTES = T::A_BYTES, STAGE_BYTES = T::STAGE_BYTES, PER_TILE = T::SLOTS_A + T::SLOTS_B;
    constexpr int WTM = BM / WAVES_M, WTN = BN / WAVES_N, TM = WTM / 32, TN = WTN / 32;
    static_assert(WAVES_M * WAVES_N == 4 && TM * TN <= 8 && TM >= 2 && PER_TILE <= 63, "one matrix wave per SIMD; at most 128 accumulator registers a lane; vmcnt is a 6-bit counter");
    static_assert(!B_KN || BN >= 128, "the [K][N] permutation moves a chunk by up to 12 places inside its row");
    extern __shared__ __align__(16) char smem[];
    stage_args(p);
    const int tid = threadIdx.x, lane = tid & 63;
    const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
    const int wm = wave % WAVES_M, wn = wave / WAVES_M;
    const unsigned long long t_entry = p.phase ? clock64() : 0ull;
    int tm_, tn_, sk_s = 0, sk_tile = 0;
    if constexpr (SK) {
        // K-slice s of tile xcd * tpx + slot is workgroup (slot * S + s) * 8 + xcd: a tile's slices share an XCD
        // (sk_finish says more).  An XCD's run of the tile order covers about as many row tiles as column tiles, so
        // its L2 pulls few panels of either operand: 1500 x 5120 -> 1280 fetched 156 MB with runs that walked whole
        // columns of 12 row tiles
        const int xcd = blockIdx.x & 7, idx = blockIdx.x >> 3;
        sk_s = idx % p.sk_S;
        sk_tile = xcd * p.sk_tpx + idx / p.sk_S;
        if (sk_tile >= p.tiles_m * p.tiles_n) return;          // the whole workgroup: the last XCD's run may be short
        const int width = p.group_m * p.tiles_n, g = sk_tile / width, in = sk_tile - g * width;
        const int first = g * p.group_m, gsz = min(p.tiles_m - first, p.group_m);
        tm_ = first + in % gsz;
        tn_ = in / gsz;
    } else {
        tile_of(p, tm_, tn_);
    }
    // (the divisions above run on the vector unit: hand the results back to scalar registers, which the direct loads'
    // base addresses have to be in)
    const int m0 = __builtin_amdgcn_readfirstlane(tm_ * BM), n0 = __builtin_amdgcn_readfirstlane(tn_ * BN);
    sk_s = __builtin_amdgcn_readfirstlane(sk_s);
    const long bz = blockIdx.y;
    const int nk = SK ? p.K / BK / p.sk_S : p.K / BK;      // the launcher guarantees whole BK-deep tiles per slice
    const long a_step = BK * 2, b_step = B_KN ? (long)BK * p.ldB * 2 : BK * 2;
    const char *Ag = reinterpret_cast<const char *>(p.A + bz * p.sA + (long)m0 * p.ldA) + (SK ? (long)sk_s * nk * a_step : 0L);
    const char *Bg = reinterpret_cast<const char *>(p.B + bz * p.sB + (B_KN ? (long)n0 : (long)n0 * p.ldB)) + (SK ? (long)sk_s * nk * b_step : 0L);
    const uint32_t lds0 = (uint32_t)(uintptr_t)(__attribute__((address_space(3))) char *)smem;
    auto barrier = [&]() {
        asm volatile("" ::: "memory");
        __builtin_amdgcn_s_barrier();
        asm volatile("" ::: "memory");
    };
    // A launch whose store the helpers can share (coop_store_applies) has eight waves, and the four that do not multiply
    // take half of it (store_coop_epi): wave 4 + w shares a SIMD with matrix wave w.
    const bool coop = !SK && blockDim.x == 512 && coop_store_applies(p);      // uniform
    constexpr int COOP_BUF = 2 * 32 * (WTN + 8) * 2;                         // a matrix wave's two staging areas
    auto help_store = [&]() {
        const int mwave = wave - 4;
        store_coop<TM, WTN, true>(p, smem + mwave * COOP_BUF, m0 + (mwave % WAVES_M) * WTM, n0 + (mwave / WAVES_M) * WTN, lane, bz,
                                  [](auto) {}, barrier);
    };
    if (wave == 4) {
        nothing_pending();
        // Per-lane offsets of the tile's 1 KB slots.  A tile that lies inside the operands needs no clamping, and its
        // slots s and s + 2 differ by a constant (eight rows of a K-contiguous operand, 64 / (BN / 8) k-rows of the
        // [K][N] one; the chunk permutation has period two in s): two offsets computed in full, the others one add
        // each -- this wave alone stands between the launch and the first request, at a vector instruction every
        // eight clocks.
        uint32_t offa[T::SLOTS_A], offb[T::SLOTS_B];
        if (m0 + BM <= p.M && n0 + BN <= (B_KN ? p.NB : p.N)) {          // uniform
            const uint32_t step_a = (uint32_t)(8 * p.ldA * 2), step_b = (uint32_t)((B_KN ? 64 / (BN / 8) : 8) * p.ldB * 2);
            const uint32_t a0 = T::a_offset(p, m0, 0, lane), a1 = T::a_offset(p, m0, 1, lane);
            const uint32_t b0 = T::b_offset(p, n0, 0, lane), b1 = T::b_offset(p, n0, 1, lane);
#pragma unroll
            for (int s = 0; s < T::SLOTS_A; s++) offa[s] = ((s & 1) ? a1 : a0) + (uint32_t)(s & ~1) * step_a;
#pragma unroll
            for (int s = 0; s < T::SLOTS_B; s++) offb[s] = ((s & 1) ? b1 : b0) + (uint32_t)(s & ~1) * step_b;
        } else {
#pragma unroll
            for (int s = 0; s < T::SLOTS_A; s++) offa[s] = T::a_offset(p, m0, s, lane);
#pragma unroll
            for (int s = 0; s < T::SLOTS_B; s++) offb[s] = T::b_offset(p, n0, s, lane);
        }
        auto request = [&](int kt, int stage) {
            const char *ab = Ag + (long)kt * a_step, *bb = Bg + (long)kt * b_step;
            const uint32_t sa = lds0 + stage * STAGE_BYTES, sb = sa + A_BYTES;
#pragma unroll
            for (int s = 0; s < T::SLOTS_A; s++) T::request(ab, offa[s], sa + s * 1024);
#pragma unroll
            for (int s = 0; s < T::SLOTS_B; s++) T::request(bb, offb[s], sb + s * 1024);
        };
        // requests complete in order: "tile t has landed" is "no more outstanding than were issued after it"
        request(0, 0);
        if (nk > 1) { request(1, 1); asm volatile("s_waitcnt vmcnt(%0)" ::"n"(PER_TILE) : "memory"); }
        else asm volatile("s_waitcnt vmcnt(0)" ::: "memory");
        barrier();                                                  // tile 0 has landed
        if (nk > 2) request(2, 2);
        for (int kt = 0; kt < nk; kt++) {
            if (kt + 2 < nk) asm volatile("s_waitcnt vmcnt(%0)" ::"n"(PER_TILE) : "memory");      // tile kt + 1 has landed
            else asm volatile("s_waitcnt vmcnt(0)" ::: "memory");
            barrier();                                              // B_kt
            if (kt + 3 < nk) request(kt + 3, kt % 3);
        }
        if (coop) help_store();
        return;
    }
    float2v *ln_slot = reinterpret_cast<float2v *>(smem + STAGES * STAGE_BYTES);
    if (wave >= 5 && !(wave == 5 && p.lnf_stats)) {
        // nothing to do beside the K loop: keep the barriers' count, then help with the store
        barrier();
        for (int kt = 0; kt < nk; kt++) barrier();
        if (coop) help_store();
        return;
    }
    if (wave == 5) {
        // the statistics wave of a folded layer norm
        lnf_stats_wave<BM, BN, true>(p, ln_slot, m0, n0, bz, lane, nk, barrier);
        if (coop) help_store();
        return;
    }

    // fragment read offsets inside a stage (bytes): rows of A, and this wave's columns of B in either layout
    const int frow = lane & 31, fhi = lane >> 5;
    const int swz = T::rowswz(lane & 15);
    int a_rd[KS], b_rd[KS], bt_rd[TN];
#pragma unroll
    for (int ks = 0; ks < KS; ks++) {
        const int cc = ((2 * ks + fhi) ^ swz) << 4;
        a_rd[ks] = (wm * WTM + frow) * ROWB + cc;
        b_rd[ks] = A_BYTES + (wn * WTN + frow) * ROWB + cc;
    }
    {
        const int kk = (lane >> 2) & 3;
#pragma unroll
        for (int i = 0; i < TN; i++) {
            const int col = (wn * WTN + i * 32 + ((lane >> 4) & 1) * 16 + (lane & 3) * 4) ^ (kk << 5);
            bt_rd[i] = A_BYTES + ((fhi * 8 + kk) * BN + col) * 2;
        }
    }
    // fragment q of a 16-deep step: q < TM the A rows 32 q .., else the wave's B columns 32 (q - TM) ..
    constexpr int NFRAG = TM + TN;
    auto read_frag = [&](const char *st, int ks, int q, half8v (&a)[TM], half8v (&b)[TN]) {
        if (q < TM) {
            a[q] = *reinterpret_cast<const half8v *>(st + a_rd[ks] + q * 32 * ROWB);
        } else if (!B_KN) {
            b[q - TM] = *reinterpret_cast<const half8v *>(st + b_rd[ks] + (q - TM) * 32 * ROWB);
        } else {
            const char *bs = st + bt_rd[q - TM] + ks * 16 * BN * 2;
            short4v lo = __builtin_amdgcn_ds_read_tr16_b64_v4i16((__attribute__((address_space(3))) short4v *)(bs));
            short4v hi = __builtin_amdgcn_ds_read_tr16_b64_v4i16((__attribute__((address_space(3))) short4v *)(bs + 4 * BN * 2));
            short8v both = {lo[0], lo[1], lo[2], lo[3], hi[0], hi[1], hi[2], hi[3]};
            b[q - TM] = __builtin_bit_cast(half8v, both);
        }
    };
    auto read_step = [&](const char *st, int ks, half8v (&a)[TM], half8v (&b)[TN]) {
#pragma unroll
        for (int q = 0; q < NFRAG; q++) read_frag(st, ks, q, a, b);
    };
    float16v acc[TN][TM];
#pragma unroll
    for (int i = 0; i < TN; i++)
#pragma unroll
        for (int j = 0; j < TM; j++)
#pragma unroll
            for (int r = 0; r < 16; r++) acc[i][j][r] = 0.0f;
    // The MFMAs of rows [JLO, JHI) x all columns of one step, from fragment set (a, b), with the reads of step ks of
    // the stage at st into set (da, db) dealt between them: a wave that issues its six or eight LDS instructions in
    // one burst stands at them while the LDS queue drains, and its matrix pipe runs dry behind it.  The scheduling
    // groups pin the order the source has: one MFMA, then the LDS reads that follow it.
    auto step = [&](auto JLO, auto JHI, const half8v (&a)[TM], const half8v (&b)[TN], const char *st, int ks, half8v (&da)[TM], half8v (&db)[TN]) {
        constexpr int jlo = decltype(JLO)::value, jhi = decltype(JHI)::value, NM = (jhi - jlo) * TN;
        static_for<NM>([&](auto Mi) {
            constexpr int m = decltype(Mi)::value, j = jlo + m / TN, i = m % TN;
            acc[i][j] = __builtin_amdgcn_mfma_f32_32x32x16_f16(b[i], a[j], acc[i][j], 0, 0, 0);
            constexpr int q0 = (m * NFRAG) / NM, q1 = ((m + 1) * NFRAG) / NM;      // fragments [q0, q1) go behind MFMA m
            static_for<q1 - q0>([&](auto Qi) { read_frag(st, ks, q0 + decltype(Qi)::value, da, db); });
        });
        static_for<NM>([&](auto Mi) {
            constexpr int m = decltype(Mi)::value, q0 = (m * NFRAG) / NM, q1 = ((m + 1) * NFRAG) / NM;
            constexpr int a_frags = (q1 < TM ? q1 : TM) - (q0 < TM ? q0 : TM), b_frags = (q1 - q0) - a_frags;
            __builtin_amdgcn_sched_group_barrier(0x008, 1, 0);
            if constexpr (q1 > q0) __builtin_amdgcn_sched_group_barrier(0x100, a_frags + b_frags * (B_KN ? 2 : 1), 0);
        });
    };
    auto mma = [&](auto JLO, auto JHI, const half8v (&a)[TM], const half8v (&b)[TN]) {
        constexpr int jlo = decltype(JLO)::value, jhi = decltype(JHI)::value;
#pragma unroll
        for (int j = jlo; j < jhi; j++)
#pragma unroll
            for (int i = 0; i < TN; i++) acc[i][j] = __builtin_amdgcn_mfma_f32_32x32x16_f16(b[i], a[j], acc[i][j], 0, 0, 0);
    };
    const bool probe = p.clk && blockIdx.x == 0 && blockIdx.y == 0 && tid == 0;
    if (probe) { p.clk[0] = clock64(); p.clk[1] = wall_clock64(); }
    const bool phases = p.phase && (int)blockIdx.x < p.phase_wgs && blockIdx.y == 0;      // uniform
    unsigned long long ph_t[4] = {0, 0, 0, t_entry};
    auto phase_mark = [&](int i) { if (phases) ph_t[i] = clock64(); };
    // Three sets of fragment registers: step s of a tile whose rotation is R sits in set (R + s) % 3, and the reads run
    // two steps ahead of the MFMAs (one step ahead, a wave's reads came back just too late: 6 KB per wave and step at the
    // 32 B/clock a SIMD takes from the LDS is 190 of the 256 clocks its eight MFMAs last, before any queueing).  Four
    // steps a tile, so the rotation advances by one per tile and the loop body is three tiles long.
    half8v fa[3][TM], fb[3][TN];
    half4v cb[TN][4];
    load_col_bias<TN, WTN>(p, cb, n0, wn, lane, bz);              // sixteen registers held through the loop; no trip to memory after it
    barrier();                                                      // tile 0 has landed
    read_step(smem, 0, fa[0], fb[0]);
    read_step(smem, 1, fa[1], fb[1]);
    int stage = 0;
    auto tile = [&](auto R, int kt) {
        constexpr int r = decltype(R)::value, s0 = r % 3, s1 = (r + 1) % 3, s2 = (r + 2) % 3;
        const char *st = smem + stage * STAGE_BYTES;
        stage = stage == STAGES - 1 ? 0 : stage + 1;
        const char *nx = smem + stage * STAGE_BYTES;
        using std::integral_constant;
        constexpr integral_constant<int, 0> J0{};
        constexpr integral_constant<int, TM / 2> JH{};
        constexpr integral_constant<int, TM> JE{};
        // steps 0 and 1, with the reads of steps 2 and 3
        step(J0, JE, fa[s0], fb[s0], st, 2, fa[s2], fb[s2]);
        __builtin_amdgcn_sched_barrier(0);
        step(J0, JE, fa[s1], fb[s1], st, 3, fa[s0], fb[s0]);
        __builtin_amdgcn_sched_barrier(0);
        // step 2: every fragment read of tile kt has returned before this wave lets the loader have the stage; the
        // reads of the next tile's steps 0 and 1 follow the barrier (past the last tile they fetch nothing anybody uses)
        asm volatile("s_waitcnt lgkmcnt(0)" ::: "memory");
        mma(J0, JH, fa[s2], fb[s2]);
        __builtin_amdgcn_sched_barrier(0);
        barrier();                                                  // B_kt
        step(JH, JE, fa[s2], fb[s2], nx, 0, fa[s1], fb[s1]);
        __builtin_amdgcn_sched_barrier(0);
        // step 3
        step(J0, JE, fa[s0], fb[s0], nx, 1, fa[s2], fb[s2]);
        __builtin_amdgcn_sched_barrier(0);
        (void)kt;
    };
    phase_mark(0);
    for (int kt = 0;;) {
        tile(std::integral_constant<int, 0>{}, kt);
        if (++kt == nk) break;
        tile(std::integral_constant<int, 1>{}, kt);
        if (++kt == nk) break;
        tile(std::integral_constant<int, 2>{}, kt);
        if (++kt == nk) break;
    }
    phase_mark(1);
    auto phase_store = [&]() {
        if (!phases) return;
        const unsigned long long issued = clock64();
        asm volatile("s_waitcnt vmcnt(0)" ::: "memory");
        const unsigned long long done = clock64();
        if (lane == 0) {
            unsigned long long *t = p.phase + ((long)blockIdx.x * 4 + wave) * 4;
            t[0] = ph_t[0] - ph_t[3]; t[1] = ph_t[1] - ph_t[0]; t[2] = issued - ph_t[1]; t[3] = done - issued;
        }
    };
    if constexpr (SK) {
        sk_finish<TM, TN, WTM, WTN, 4, STAGES * STAGE_BYTES>(p, acc, cb, smem, sk_tile, sk_s, m0, n0, wm, wn, wave, lane, bz);
        phase_store();
        if (probe) { p.clk[2] = clock64(); p.clk[3] = wall_clock64(); }
        return;
    }
    LnFold<TM> ln;
    if (p.lnf_stats) {
        ln.on = true; ln.col = reinterpret_cast<const float *>(ln_slot + BM); ln.bn = BN;
#pragma unroll
        for (int j = 0; j < TM; j++) { const float2v v = ln_slot[wm * WTM + 32 * j + (lane & 31)]; ln.r[j] = v[0]; ln.rmu[j] = v[1]; }
    }
    if (coop) {
#pragma unroll
        for (int i = 0; i < TN; i++)
#pragma unroll
            for (int g = 0; g < 4; g++) asm volatile("" ::"v"(cb[i][g]));      // in registers ahead of the first store (store_tile_simple)
        char *buf = smem + wave * COOP_BUF;
        store_coop<TM, WTN, false>(p, buf, m0 + wm * WTM, n0 + wn * WTN, lane, bz,
                                   [&](auto J) { constexpr int j = decltype(J)::value; stage_block<j, TM, TN, WTN>(acc, cb, ln, wn, buf + (j & 1) * (COOP_BUF / 2), lane); },
                                   barrier);
    } else {
        store_tile<TM, TN, WTM, WTN, 4, STAGES * STAGE_BYTES>(p, acc, cb, smem, m0, n0, wm, wn, wave, lane, bz, ln);
    }
    phase_store();
    if (probe) { p.clk[2] = clock64(); p.clk[3] = wall_clock64(); }
}

// Split-K epilogue: out = epi(round(sum_s part[s] + bias)) (+ residual), four columns per thread.
// The counterpart of mm_epilogue_kernel! (matmul.jl:192-217): the planes are fp32 M x N.
__global__ void splitk_epilogue_kernel(GemmArgs p, const float *part, int nsplit) {
    const long idx = ((long)blockIdx.x * blockDim.x + threadIdx.x) * 4;
    const long total = (long)p.M * p.N;
    if (idx >= total) return;
    const int n = (int)(idx % p.N), m = (int)(idx / p.N);
    float4v v = *reinterpret_cast<const float4v *>(part + idx);
    for (int s = 1; s < nsplit; s++) {
        float4v w = *reinterpret_cast<const float4v *>(part + (long)s * total + idx);
#pragma unroll
        for (int e = 0; e < 4; e++) v[e] += w[e];
    }
#pragma unroll
    for (int e = 0; e < 4; e++)
        v[e] += p.bias_mode == MI_BIAS_COL ? (float)p.bias[n + e] : p.bias_mode == MI_BIAS_ROW ? (float)p.bias[m] : 0.0f;
    const long off = (long)m * p.ldY + n;
    if (p.out_f32) {
#pragma unroll
        for (int e = 0; e < 4; e++) reinterpret_cast<float *>(p.Y)[off + e] = apply_epi(v[e], p.epi);
    } else {
        half4v o;
#pragma unroll
        for (int e = 0; e < 4; e++) o[e] = (half_t)apply_epi((float)(half_t)v[e], p.epi);
        if (p.residual) {
#pragma unroll
            for (int e = 0; e < 4; e++) o[e] = (half_t)((float)o[e] + (float)p.residual[off + e]);
        }
        if (p.clamp > 0.0f) {
#pragma unroll
            for (int e = 0; e < 4; e++) o[e] = (half_t)fminf(fmaxf((float)o[e], -p.clamp), p.clamp);
        }
        if (p.vec_store) *reinterpret_cast<half4v *>(reinterpret_cast<half_t *>(p.Y) + off) = o;
        else {
#pragma unroll
            for (int e = 0; e < 4; e++) reinterpret_cast<half_t *>(p.Y)[off + e] = o[e];
        }
    }
}

// The same sums, bias, activation and residual as splitk_epilogue_kernel, one wave per output row, followed by the
// layer norm of that row into p.lnout: lane and chunk order, summation order and rounding are those of
// layernorm_vec_kernel, so Y and lnout carry the bits the two separate launches would have written.
template <int NCH>
__global__ __launch_bounds__(256) void splitk_epilogue_ln_kernel(GemmArgs p, const float *part, int nsplit) {
    const int lane = threadIdx.x & 63, wave = threadIdx.x >> 6;
    const long m = (long)blockIdx.x * 4 + wave;
    if (m >= p.M) return;
    const long total = (long)p.M * p.N;
    const u32x4 z = {0u, 0u, 0u, 0u};
    u32x4 graw[NCH], braw[NCH];
#pragma unroll
    for (int i = 0; i < NCH; i++) {
        const int e0 = (lane + 64 * i) * 8;
        graw[i] = (p.lnout_gamma && e0 < p.N) ? ldg16(p.lnout_gamma + e0) : z;
        braw[i] = (p.lnout_beta && e0 < p.N) ? ldg16(p.lnout_beta + e0) : z;
    }
    float x[NCH][8];
    float s = 0.0f;
#pragma unroll
    for (int i = 0; i < NCH; i++) {
        const int e0 = (lane + 64 * i) * 8;
        if (e0 < p.N) {
            const float *pp = part + m * p.N + e0;
            float4v v0 = *reinterpret_cast<const float4v *>(pp), v1 = *reinterpret_cast<const float4v *>(pp + 4);
            for (int sp = 1; sp < nsplit; sp++) {
                const float4v w0 = *reinterpret_cast<const float4v *>(pp + (long)sp * total), w1 = *reinterpret_cast<const float4v *>(pp + (long)sp * total + 4);
#pragma unroll
                for (int e = 0; e < 4; e++) { v0[e] += w0[e]; v1[e] += w1[e]; }
            }
            const long off = m * p.ldY + e0;
            half8v o;
#pragma unroll
            for (int e = 0; e < 8; e++) {
                float v = e < 4 ? v0[e] : v1[e - 4];
                v += p.bias_mode == MI_BIAS_COL ? (float)p.bias[e0 + e] : p.bias_mode == MI_BIAS_ROW ? (float)p.bias[m] : 0.0f;
                o[e] = (half_t)apply_epi((float)(half_t)v, p.epi);
            }
            if (p.residual) {
                const half8v rv = as_half8(ldg16(p.residual + off));
#pragma unroll
                for (int e = 0; e < 8; e++) o[e] = (half_t)((float)o[e] + (float)rv[e]);
            }
            if (p.clamp > 0.0f) {
#pragma unroll
                for (int e = 0; e < 8; e++) o[e] = (half_t)fminf(fmaxf((float)o[e], -p.clamp), p.clamp);
            }
            *reinterpret_cast<half8v *>(reinterpret_cast<half_t *>(p.Y) + off) = o;
#pragma unroll
            for (int j = 0; j < 8; j++) { x[i][j] = (float)o[j]; s += x[i][j]; }
        } else {
#pragma unroll
            for (int j = 0; j < 8; j++) x[i][j] = 0.0f;
        }
    }
    s = wave_sum(s);
    const float mu = s / (float)p.N;
    float s2 = 0.0f;
#pragma unroll
    for (int i = 0; i < NCH; i++) {
        if ((lane + 64 * i) * 8 < p.N) {
#pragma unroll
            for (int j = 0; j < 8; j++) { const float d = x[i][j] - mu; s2 = fmaf(d, d, s2); }
        }
    }
    s2 = wave_sum(s2);
    const float r = 1.0f / sqrtf(s2 / (float)p.N + p.lnout_eps);
#pragma unroll
    for (int i = 0; i < NCH; i++) {
        const int e0 = (lane + 64 * i) * 8;
        if (e0 < p.N) {
            const half8v gv = as_half8(graw[i]), bv = as_half8(braw[i]);
            half8v o;
#pragma unroll
            for (int j = 0; j < 8; j++)
                o[j] = ln_norm1(x[i][j], mu, r, p.lnout_gamma != nullptr, p.lnout_gamma ? (float)gv[j] : 0.0f, p.lnout_beta != nullptr, p.lnout_beta ? (float)bv[j] : 0.0f);
            *reinterpret_cast<half8v *>(p.lnout + m * p.N + e0) = o;
        }
    }
}

// ------------------------------------------------------------------------------------------
bool g_ready = false;
int g_cus = 256;
// Inside mi_*_plan_caps the planners answer for the device the caller describes instead of the one they run on.
thread_local int tl_plan_cus = 0;          // > 0: compute units to plan for
thread_local bool tl_plan_mfma = true;     // false: the described device has no matrix unit
unsigned long long *g_clock_probe = nullptr;      // mi_set_clock_probe
unsigned long long *g_phase_probe = nullptr;      // mi_set_phase_probe
int g_phase_wgs = 0;

// Scratch of mi_gemm_f16_noalloc: every GPU the library runs on holds its own copy of this array, at its own
// address, until the process ends.  Host code never uses the name as a pointer; g_scratch_ptr[device] is the
// address hipGetSymbolAddress gave with that device current.
constexpr int MAX_DEVICES = 64;
void *g_scratch_ptr[MAX_DEVICES] = {};

unsigned *g_sk_flags_ptr[MAX_DEVICES] = {};
unsigned *g_status_ptr[MAX_DEVICES] = {};    // the device's copy of device_status_words
int g_sk_state[MAX_DEVICES] = {};            // 0: not probed, 1: usable, -1: this device does not deal workgroups round robin
std::atomic<unsigned> g_sk_epoch{0};
std::atomic<bool> g_sk_enabled{true};        // mi_set_in_launch_exchange
constexpr int SK_SPIN_DEFAULT = 1 << 18;     // polls of a few hundred ns each: a partner that has not shown up after ~0.1 s will not
int g_sk_spin = SK_SPIN_DEFAULT;             // mi_test_exchange_faults
unsigned g_sk_pub_xor = 0, g_sk_xcc_xor = 0;

// Workgroup -> XCD: every workgroup of a 1024-workgroup probe writes the id of the XCD it runs on (HW_REG_XCC_ID).
__global__ void xcc_probe_kernel(unsigned *out) {
    if (threadIdx.x == 0) out[blockIdx.x] = __builtin_amdgcn_s_getreg((3 << 11) | 20);      // XCC_ID, bits 3:0
}

// The split-K peer reduction relies on workgroups pid, pid + 8, pid + 16, ... sharing an XCD (one L2).  Checked once
// per device on a probe launch: all workgroups with the same pid % 8 must report one XCD.  Uses the flag words as the
// probe's output (they are zeroed again) and synchronises the device: call from mi_init only.
int sk_probe_current_device() {
    int dev = -1;
    if (hipGetDevice(&dev) != hipSuccess || dev < 0 || dev >= MAX_DEVICES) return -1;
    if (g_sk_state[dev]) return g_sk_state[dev];
    void *ptr = nullptr, *sptr = nullptr;
    if (hipGetSymbolAddress(&sptr, HIP_SYMBOL(device_status_words)) != hipSuccess || !sptr) return g_sk_state[dev] = -1;
    g_status_ptr[dev] = reinterpret_cast<unsigned *>(sptr);
    if (hipGetSymbolAddress(&ptr, HIP_SYMBOL(sk_flag_words)) != hipSuccess || !ptr) return g_sk_state[dev] = -1;
    g_sk_flags_ptr[dev] = reinterpret_cast<unsigned *>(ptr);
    constexpr int NP = 1024;
    static_assert(NP <= SK_BANKS * SK_FLAGS, "probe output fits the flag words");
    unsigned host[NP];
    hipLaunchKernelGGL(xcc_probe_kernel, dim3(NP), dim3(64), 0, 0, g_sk_flags_ptr[dev]);
    bool ok = hipGetLastError() == hipSuccess && hipMemcpy(host, g_sk_flags_ptr[dev], sizeof(host), hipMemcpyDeviceToHost) == hipSuccess;
    ok = ok && hipMemset(g_sk_flags_ptr[dev], 0, sizeof(host)) == hipSuccess && hipDeviceSynchronize() == hipSuccess;
    for (int i = 8; ok && i < NP; i++) ok = host[i] == host[i & 7];
    return g_sk_state[dev] = ok ? 1 : -1;
}
bool sk_usable() {
    int dev = -1;
    return g_sk_enabled.load() && hipGetDevice(&dev) == hipSuccess && dev >= 0 && dev < MAX_DEVICES && g_sk_state[dev] == 1;
}

// The current device's copy of `scratch`; resolved once per device, with that device current.  Null on failure.
void *scratch_of_current_device() {
    int dev = -1;
    if (hipGetDevice(&dev) != hipSuccess || dev < 0 || dev >= MAX_DEVICES) return nullptr;
    if (!g_scratch_ptr[dev]) {
        void *ptr = nullptr;
        if (hipGetSymbolAddress(&ptr, HIP_SYMBOL(scratch)) != hipSuccess) return nullptr;
        g_scratch_ptr[dev] = ptr;
    }
    return g_scratch_ptr[dev];
}

// LDS of the four-wave kernel: three 64-deep stages of both operands (the store's staging reuses them), then a folded
// layer norm's (r, r mu) per row and colsum and biasp per column
template <int BM, int BN>
constexpr int w4_lds_bytes() { return 3 * (BM + BN) * 64 * 2 + BM * 8 + BN * 8; }


bool mfma_addressable(const GemmArgs &a, bool b_kn) {
    if (a.K % 8 || a.ldA % 8 || a.ldB % 8 || a.sA % 8 || a.sB % 8) return false;
    if (!aligned_to(a.A, 16) || !aligned_to(a.B, 16)) return false;
    if (b_kn && (a.NB % 8 || a.NB < 8 || a.NB < a.N)) return false;
    if (a.bias && a.bias_mode == MI_BIAS_COL && !aligned_to(a.bias, 8)) return false;
    return a.M >= 1 && a.N >= 1 && a.K >= 8;
}

template <int BM, int BN, int WM, int WN>
int launch_w4(GemmArgs a, bool b_kn, int64_t nbatch, hipStream_t st) {
    if (a.K < 64 || a.K % 64 || a.ag.x) return MI_DECLINE_EXTENT;
    set_tiles(a, BM, BN);
    a.vec_store = rows_vec16(a);
    // per-lane load offsets are 32-bit byte offsets from the tile origin
    if ((int64_t)BM * a.ldA * 2 >= (1ll << 31) || (int64_t)(b_kn ? 64 : BN) * a.ldB * 2 >= (1ll << 31)) return MI_DECLINE_EXTENT;
    a.clk = g_clock_probe;
    a.phase = g_phase_probe; a.phase_wgs = g_phase_wgs;
    dim3 grid((unsigned)(a.tiles_m * a.tiles_n), (unsigned)nbatch);
    constexpr int lds = w4_lds_bytes<BM, BN>();
    // four matrix waves and the loader, plus the statistics wave of a folded layer norm; eight waves when the four that
    // do not multiply can help with the store
    const dim3 block(coop_store_applies(a) ? 512 : a.lnf_stats ? 384 : 320);
    if (b_kn) hipLaunchKernelGGL((gemm_w4_kernel<BM, BN, WM, WN, true>), grid, block, lds, st, a);
    else      hipLaunchKernelGGL((gemm_w4_kernel<BM, BN, WM, WN, false>), grid, block, lds, st, a);
    return hipGetLastError() == hipSuccess ? MI_OK : MI_ERROR_LAUNCH;
}

bool sk_fits(int64_t M, int64_t N, int64_t K, int bm, int bn, int split);

// The four-wave kernel with two workgroups per 128 x 128 tile exchanging their partial tiles.
int launch_w4_peer(GemmArgs a, bool b_kn, int split, void *ws, hipStream_t st) {
    constexpr int BM = 128, BN = 128;
    if (a.ag.x || split != 2 || !sk_usable() || !sk_fits(a.M, a.N, a.K, BM, BN, split)) return MI_DECLINE_EXTENT;
    int dev = 0;
    if (hipGetDevice(&dev) != hipSuccess) return MI_ERROR_DEVICE;
    a.tiles_m = (int)ceil_div(a.M, BM);
    a.tiles_n = (int)ceil_div(a.N, BN);
    a.group_m = 1;
    while (a.group_m * a.group_m < (int)ceil_div((int64_t)a.tiles_m * a.tiles_n, 8) && a.group_m < a.tiles_m) a.group_m++;
    a.vec_store = rows_vec16(a);
    if ((int64_t)BM * a.ldA * 2 >= (1ll << 31) || (int64_t)(b_kn ? 64 : BN) * a.ldB * 2 >= (1ll << 31)) return MI_DECLINE_EXTENT;
    const int tiles = a.tiles_m * a.tiles_n;
    a.sk_S = split;
    a.sk_tpx = (int)ceil_div(tiles, 8);
    a.sk_part = reinterpret_cast<float *>(ws);
    const unsigned launch = ++g_sk_epoch;
    a.sk_epoch = sk::epoch_of(launch);
    a.sk_flags = g_sk_flags_ptr[dev] + (size_t)(launch % SK_BANKS) * SK_FLAGS;
    a.sk_spin = g_sk_spin; a.sk_pub_xor = g_sk_pub_xor; a.sk_xcc_xor = g_sk_xcc_xor;
    a.status = g_status_ptr[dev];
    a.clk = g_clock_probe;
    a.phase = g_phase_probe; a.phase_wgs = g_phase_wgs;
    dim3 grid((unsigned)(8 * a.sk_tpx * split), 1);
    constexpr int lds = w4_lds_bytes<BM, BN>();
    if (b_kn) hipLaunchKernelGGL((gemm_w4_kernel<BM, BN, 2, 2, true, true>), grid, dim3(320), lds, st, a);
    else      hipLaunchKernelGGL((gemm_w4_kernel<BM, BN, 2, 2, false, true>), grid, dim3(320), lds, st, a);
    return hipGetLastError() == hipSuccess ? MI_OK : MI_ERROR_LAUNCH;
}

constexpr int RING_TILE = 5, DEEP_TILE = 6, DEEP_SERIAL_TILE = 7;      // indices into TILE_MODELS: gemm_ring_kernel, gemm_deep_kernel with four matrix waves and one
// tile: index into TILE_MODELS.  The four-wave kernel takes ordinary operands in whole 64-deep tiles only; a gathered operand
// (implicit-GEMM convolution) or a K % 64 planned onto one of its tiles runs the pipelined kernel's same tile instead: same K order per
// output, same bits.  On the ring a gathered operand runs the pipelined 64 x 64 tile, whose order of a long K is not the ring's; the 32 x 32
// tiles are not planned for one.
int launch_tile(int tile, const GemmArgs &a, bool b_kn, int64_t nbatch, hipStream_t st) {
    const bool plain = !a.ag.x && a.K % 64 == 0;
    switch (tile) {
        case 0: return plain ? launch_w4<128, 256, 1, 4>(a, b_kn, nbatch, st) : mi_pipe_launch(0, a, b_kn, nbatch, st);
        case 1: return plain ? launch_w4<192, 128, 2, 2>(a, b_kn, nbatch, st) : mi_pipe_launch(1, a, b_kn, nbatch, st);
        case RING_TILE:
            if (!a.ag.x) {
                const int rc = mi_ring_launch(a, b_kn, nbatch, st);
                if (rc != MI_DECLINE_EXTENT) return rc;     // declined: a row pitch beyond its 32-bit offsets
            }
            return mi_pipe_launch(4, a, b_kn, nbatch, st);
        case DEEP_TILE:
        case DEEP_SERIAL_TILE:
            if (!a.ag.x) {
                const int rc = mi_deep_launch(a, tile == DEEP_TILE, b_kn, nbatch, st);
                if (rc != MI_DECLINE_EXTENT) return rc;
            }
            return mi_pipe_launch(4, a, b_kn, nbatch, st);
        default: return mi_pipe_launch(tile, a, b_kn, nbatch, st);
    }
}

// Tile and K-split of a pipelined GEMM, chosen by estimated time: launch + prologue/store + (K / 64) steps, where a step costs
// step_lo when few workgroups run, rises linearly to step_full when every CU holds one (clock and memory give way under
// load), and beyond that grows with the number of rounds of CUs-many workgroups (by `round`, below 1 where co-resident
// workgroups overlap).  A K that ends inside a tile makes every step `tail` times as long: its rows are no multiple of
// a cache line, so most 128-byte pieces of them touch two.  A GELU store adds `gelu` a round.  A split adds the second
// launch (4.4 us) and the fp32 planes (0.38 us per MB).
// Fitted to every tile timed on 260 shapes in a replayed graph (M 9..8192, N 64..8192, K 72..5120, both layouts, a third of
// them with K % 64, a third with GELU).  On these the cheapest estimate lands within 0.4 % of the best measured tile on average,
// 15 % at worst (259 x 1728 -> 3584 with GELU).  The 32 x 32 tiles, at most one workgroup a CU, were fitted to 300 more (M 9..2048,
// N 64..5120, K 72..8192): 18 % above the best tile on average without them, 1.2 % with them.  A K that mi_ln_gemm_f16 takes, up to
// MI_LNA_KMAX, keeps one chain of sums an element: that call gives the bits of a norm followed by this GEMM, on whichever tile.
// What it replaced sent every K % 64 to 64 x 64 tiles: 1544 x 1288 -> 1288 with residual 19.8 -> 15.4 us on 128 x 128,
// 636 x 4392 -> 104 23.2 -> 13.8 on the ring, 2237 x 5096 -> 2440 with GELU 143 -> 80 on 192 x 128.
struct TileModel { int bm, bn; double step_lo, step_full, round, fixed, gelu, tail; };
constexpr int NTILES = 8;
constexpr TileModel TILE_MODELS[NTILES] = {
    {128, 256, 0.453, 0.746, 1.02, 6.1, 2.89, 1.41},
    {192, 128, 0.369, 0.613, 1.03, 5.19, 2.17, 1.38},
    {128, 128, 0.457, 0.568, 1.09, 4.27, 1.86, 1.13},
    {64, 128, 0.315, 0.394, 0.841, 3.47, 0.946, 1.17},
    {64, 64, 0.267, 0.302, 0.632, 3.04, 0.423, 1.2},
    {64, 64, 0.135, 0.22, 0.818, 3.28, 0.362, 1.3},      // gemm_ring_kernel
    {32, 32, 0.0857, 0.132, 0.624, 3.15, 0.508, 1.21},   // gemm_deep_kernel, K split over its waves
    {32, 32, 0.142, 0.112, 0.8, 3.14, 0.409, 1.15},      // gemm_deep_kernel, one chain of sums
};
constexpr int64_t RING_WGS_PER_CU = 11, DEEP_WGS = 256;      // as many as the fits have seen
// A folded norm costs the four-wave kernel, which gives it a wave beside the K loop, more than the pipelined kernel, whose threads take the
// statistics in before it, where other kernels' weights come between.  Three blocks of 64 to 1500 tokens, 384 to 1280 wide (35 stacks,
// replayed): 572 x 1280 235 -> 223 us with this, 1100 x 1024 259 -> 252, the others within 1 %.
constexpr double LNF_W4_US = 3.0;
struct TilePlan { int tile, split; bool peer; double us; };      // peer: the K-slices exchange partial tiles in the kernel (no planes)

double tile_cost_us(int64_t M, int64_t N, int64_t K, int64_t nbatch, int tile, int split, bool gelu = false) {
    const TileModel &t = TILE_MODELS[tile];
    const double cus = (double)mi_num_cus();
    const int64_t wg = ceil_div(M, t.bm) * ceil_div(N, t.bn) * nbatch * split;
    const int64_t rounds = ceil_div(wg, (int64_t)mi_num_cus());
    const double load = wg < mi_num_cus() ? (double)wg / cus : 1.0;
    const double step = (wg <= mi_num_cus() ? t.step_lo + (t.step_full - t.step_lo) * load : t.step_full * t.round * (double)rounds) * (K % 64 ? t.tail : 1.0);
    double us = 2.0 + (t.fixed - 2.0) * (1.0 + 0.8 * (double)(rounds - 1)) + (t.fixed - 2.0) * 0.4 * load + (double)((K + 63) / 64 / split) * step;
    if (split > 1) us += 4.4 + 0.38 * (double)split * (double)M * (double)N * 4.0 / 1e6;
    if (gelu) us += t.gelu * (wg > mi_num_cus() ? (double)wg / cus : 1.0);
    return us;
}

// Split-K with the partials exchanged inside the launch (four-wave kernel, 128 x 128 tiles in two K-slices, every
// workgroup resident at once): the tile's own estimate at that many workgroups, no planes and no second launch, plus
// the exchange.  A workgroup writes and reads half of its accumulators; what that costs is set by how fast the burst
// drains -- 7.7 MB from 120 or 240 workgroups take 2 to 3 us end to end.
constexpr int SK_TILE = 2;               // index into TILE_MODELS: 128 x 128
double sk_exchange_us(int64_t wg, int bm, int bn) {
    const double mb = (double)wg * bm * bn * 4.0 * 0.5 / 1e6;
    return 2.0 + 0.3 * mb;               // fitted: 29.8 us measured on 1500 x 5120 -> 1280, 22.1 on 512 x 5120 -> 1280
}
size_t sk_workspace_bytes(int64_t M, int64_t N, int bm, int bn, int split) { return (size_t)(ceil_div(M, bm) * ceil_div(N, bn)) * split * bm * bn * 4; }
bool sk_fits(int64_t M, int64_t N, int64_t K, int bm, int bn, int split) {
    const int64_t tiles = ceil_div(M, bm) * ceil_div(N, bn), tpx = ceil_div(tiles, 8);
    return split == 2 && bm == 128 && bn == 128 && K % 128 == 0 && K / 2 >= 128 && 8 * tpx * 2 <= mi_num_cus() && 8 * tpx * 2 * 8 <= SK_FLAGS;
}
// Before mi_init (planner queries without a device) the path is assumed: a workspace sized for it also holds the planes
// the same split falls back to.
bool sk_planned() {
    int dev = -1;
    if (!g_sk_enabled.load()) return false;
    if (hipGetDevice(&dev) != hipSuccess || dev < 0 || dev >= MAX_DEVICES) return true;
    return g_sk_state[dev] != -1;
}
double sk_cost_us(int64_t M, int64_t N, int64_t K, int tile, int split) {
    constexpr double step_lo = 0.428, step_full = 0.600, fixed = 4.0;        // of the four-wave kernel's 128 x 128 tile
    const TileModel &t = TILE_MODELS[tile];
    const int64_t wg = ceil_div(M, t.bm) * ceil_div(N, t.bn) * split;
    const double load = (double)wg / (double)mi_num_cus();
    const double step = step_lo + (step_full - step_lo) * load;
    return 0.9 * (2.0 + (fixed - 2.0) * (0.4 + 0.6 / (double)split) + (fixed - 2.0) * 0.4 * load + (double)(K / (64 * split)) * step +
           sk_exchange_us(wg, t.bm, t.bn));        // 0.9: 17.1 us at 1500 x 3072 -> 768, 27.9 at 1370 x 5120 -> 1280
}

// Tiles that sum a long K in an order of their own: several chains an element (gemm_ring_kernel, gemm_deep_kernel).
bool own_order(int tile, int64_t K) { return K > MI_LNA_KMAX && (tile == RING_TILE || tile == DEEP_TILE); }

// The plan depends on the extents, and on whether the operand is gathered (no 32 x 32 tiles there) and a norm folded: calls alike in
// these give the same bits whichever entry point issues them.  Up to K = MI_LNA_KMAX all unsplit calls do.
TilePlan estimate_tiles(int64_t M, int64_t N, int64_t K, int64_t nbatch, bool may_split, bool gelu, bool deep, bool lnf) {
    TilePlan best = {4, 1, false, 0.0};
    double best_us = 1e30;
    const int max_split = (may_split && nbatch == 1 && M > 8 && N % 4 == 0 && K % 64 == 0) ? 8 : 1;
    for (int split = 1; split <= max_split; split++) {
        if (split > 1 && (K % (64 * split) != 0 || K / split < 128)) continue;
        // planes that mi_gemm_f16_noalloc has room for: a call is not refused there because its estimate moved
        const bool planes = split == 1 || (double)split * (double)M * (double)N * 4.0 <= (double)MI_NOALLOC_SCRATCH_BYTES;
        for (int tile = 0; planes && tile < NTILES; tile++) {
            if (tile == RING_TILE && split > 1 && K / split <= MI_LNA_KMAX) continue;      // (a slice would be one chain)
            if (tile == RING_TILE && ceil_div(M, 64) * ceil_div(N, 64) * nbatch * split > RING_WGS_PER_CU * mi_num_cus()) continue;
            if (tile == DEEP_TILE || tile == DEEP_SERIAL_TILE) {
                if (!deep || (K > MI_LNA_KMAX) != (tile == DEEP_TILE)) continue;
                if (ceil_div(M, 32) * ceil_div(N, 32) * nbatch * split > std::min(DEEP_WGS, (int64_t)mi_num_cus())) continue;
            }
            if (gelu && own_order(tile, K)) continue;
            const double us = tile_cost_us(M, N, K, nbatch, tile, split, gelu) + (lnf && tile <= 1 ? LNF_W4_US : 0.0);
            if (us < best_us) { best_us = us; best = {tile, split, false, us}; }
        }
        if (max_split > 1 && sk_planned()) {
            if (sk_fits(M, N, K, TILE_MODELS[SK_TILE].bm, TILE_MODELS[SK_TILE].bn, split)) {
                const double us = sk_cost_us(M, N, K, SK_TILE, split);
                if (us < best_us) { best_us = us; best = {SK_TILE, split, true, us}; }
            }
        }
    }
    return best;
}

// The estimate of every tile and split takes the host about 2 us, twice a call (workspace, launch): a small table per
// thread keeps the last answers.  The key holds everything the estimate reads; flags tell places apart, as one call asks under several.
TilePlan plan_tiles(int64_t M, int64_t N, int64_t K, int64_t nbatch, bool may_split, bool gelu = false, bool deep = true, bool lnf = false) {
    struct Entry { int64_t M, N, K, nbatch; int cus, flags; TilePlan plan; };
    static thread_local Entry table[256] = {};
    const int cus = mi_num_cus(), flags = 1 | (may_split ? 2 : 0) | (may_split && sk_planned() ? 4 : 0) | (gelu ? 8 : 0) | (deep ? 16 : 0) | (lnf ? 32 : 0);
    const uint64_t h = ((uint64_t)M * 0x9E3779B97F4A7C15ull) ^ ((uint64_t)N * 0xC2B2AE3D27D4EB4Full) ^ ((uint64_t)K * 0x165667B19E3779F9ull) ^ ((uint64_t)nbatch << 17) ^ (uint64_t)flags << 32;
    Entry &e = table[(h >> 32) & 255];
    if (e.flags != flags || e.M != M || e.N != N || e.K != K || e.nbatch != nbatch || e.cus != cus)
        e = {M, N, K, nbatch, cus, flags, estimate_tiles(M, N, K, nbatch, may_split, gelu, deep, lnf)};
    return e.plan;
}

// A second look at a call that was given one of the four-wave kernel's tiles.  Against them the 128 x 128 and 64 x 128 tiles are
// estimated too high, and a residual costs the four-wave kernel more: its stores then have no helper waves, and fetch.  The
// tiles here sum K in one order, so the bits stay.  (Lowered for all calls, these estimates take some from the ring and cost stacks of
// blocks 2 to 3 %.)  2012 x 1280 -> 1152 15.6 -> 14.0 us, with residual 17.4 -> 14.9; 2791 x 512 -> 4096 with residual 29.3 -> 24.6.
//
// By how much too high: 9 % from K = 256 to 1023, and with a residual below that too (85 calls with one 0.72 to 0.97 of the four-wave
// tiles' time).  Without one the 128 x 128 tiles are as good as estimated at K = 128 and 192 (35 calls that 9 % moved were 1 to 9 % slower:
// 4525 x 192 -> 1688 9.7 -> 10.5 us, 1808 x 128 -> 3952 9.3 -> 9.95), the 64 x 128 ones lower (24 calls 0.82 to 0.95).  From K = 1024 on
// only the 128 x 128 tiles of at most one workgroup a CU are (0.85 to 1.0, one in ten 1.02 to 1.08; with residual 0.81 to 1.0): the others
// are taken where those pass 256 or 512 by a few (1571 x 1024 -> 2544 15.0 -> 16.0, 3379 x 2048 -> 2360 44 -> 49, with residual 47 -> 52).  The
// 64 x 128 ones are not from K = 768 on without a residual (1181 x 896 -> 3264 12.7 -> 14.0, 4665 x 896 -> 784 13.1 -> 14.4).
//
// What the residual costs the four-wave kernel: 2 us, and 0.6 where it has at most one workgroup a CU and K >= 256, whose tiles
// are not estimated as much too high (24 such calls, both layouts: 0.97 of the time with 2 us; 6263 x 384 -> 952 15.2 -> 13.6 us,
// 4942 x 512 -> 1032 14.95 -> 13.4.  60 of more workgroups lose 1 % with 1 us; K = 128 and 192 keep the gain at one workgroup a CU: 3470 x 192
// -> 1600 10.0 -> 8.65).  With [K][F] weights the same factors hold: 200 calls are 0.4 % above the faster side, 11 % at worst.
double estimated_high(int tile, const GemmArgs &a, int64_t wgs) {
    const bool residual = a.residual != nullptr;
    if (tile <= 1) return 1.0;
    if (a.K >= 1024) return tile == 2 && wgs <= mi_num_cus() ? (residual ? 0.91 : 0.93) : 1.0;
    if (tile == 3 && a.K >= 768 && !residual) return 1.0;
    return residual || a.K >= 256 ? 0.91 : tile == 2 ? 0.97 : 0.92;
}
int settled_tile(int tile, const GemmArgs &a, int64_t nbatch) {
    if (tile > 1 || a.ag.x || a.K % 64 || a.lnf_stats || a.stats_out || a.epi == MI_EPI_GELU_ERF || a.epi == MI_EPI_GELU_TANH) return tile;
    double best = 1e30;
    for (int t = 0; t < 4; t++) {
        const int64_t wgs = ceil_div(a.M, TILE_MODELS[t].bm) * ceil_div(a.N, TILE_MODELS[t].bn) * nbatch;
        if (t > 1 && a.K >= 1024 && wgs > 2 * mi_num_cus()) continue;      // (nor does a residual make up for theirs)
        const double us = tile_cost_us(a.M, a.N, a.K, nbatch, t, 1) * estimated_high(t, a, wgs) + (t <= 1 && a.residual ? (a.K >= 256 && wgs <= mi_num_cus() ? 0.6 : 2.0) : 0.0);
        if (us < best) { best = us; tile = t; }
    }
    return tile;
}

// Workspace of a planned split: the planes, or the exchanged partials of the peer reduction (never less than the planes,
// so a launch that cannot take the peer path -- a gathered operand -- falls back to planes in the same workspace).
size_t plan_workspace_bytes(const TilePlan &tp, int64_t M, int64_t N) {
    if (tp.split <= 1) return 0;
    return round_up(tp.peer ? sk_workspace_bytes(M, N, TILE_MODELS[tp.tile].bm, TILE_MODELS[tp.tile].bn, tp.split) : (size_t)tp.split * M * N * sizeof(float), 256);
}

// Workspace to ask for: of the plan, and of the plan without the 32 x 32 tiles -- a gathered operand's, and the size that recorded
// plans and callers' buffers had before those tiles.
size_t planned_workspace(int64_t M, int64_t N, int64_t K) {
    return std::max(plan_workspace_bytes(plan_tiles(M, N, K, 1, true), M, N), plan_workspace_bytes(plan_tiles(M, N, K, 1, true, false, false), M, N));
}

int gemm_path(const GemmArgs &a, bool b_kn, int64_t nbatch) {
    if (a.M < 1 || a.N < 1 || a.K < 1) return MI_GEMM_DECLINE;
    bool addr = mfma_addressable(a, b_kn);
    if (a.M <= 8 && nbatch == 1 && addr && (b_kn || (size_t)8 * a.K * sizeof(half_t) <= SKINNY_FK_LDS_MAX)) return MI_GEMM_SKINNY;
    if (addr && tl_plan_mfma) return MI_GEMM_MFMA;
    return MI_GEMM_SCALAR;
}

int fill_args(GemmArgs &a, void *Y, const void *X, const void *W, const void *bias, const void *residual,
              int64_t T, int64_t K, int64_t F, int64_t ldY, int64_t ldX, int64_t ldW,
              int w_layout, int bias_mode, int epi, int out_dtype, int64_t sY, int64_t sX, int64_t sW, int64_t sBias = 0) {
    if (!Y || !X || !W) return MI_DECLINE_OPERANDS;
    if (T < 0 || K < 0 || F < 0 || T > INT32_MAX || K > INT32_MAX || F > INT32_MAX) return MI_DECLINE_EXTENT;
    if (w_layout != MI_W_KF && w_layout != MI_W_FK) return MI_DECLINE_OPERANDS;
    if (out_dtype != MI_F16 && out_dtype != MI_F32) return MI_DECLINE_OPERANDS;
    if (epi < MI_EPI_NONE || epi > MI_EPI_RELU) return MI_DECLINE_UNSUPPORTED;
    if (bias_mode < MI_BIAS_NONE || bias_mode > MI_BIAS_ROW) return MI_DECLINE_BIAS;
    if (bias_mode != MI_BIAS_NONE && !bias) return MI_DECLINE_BIAS;
    if (residual && out_dtype != MI_F16) return MI_DECLINE_UNSUPPORTED;
    if (ldX < K || ldY < F || ldW < (w_layout == MI_W_KF ? F : K)) return MI_DECLINE_EXTENT;
    a.Y = Y; a.A = (const half_t *)X; a.B = (const half_t *)W;
    a.bias = bias_mode == MI_BIAS_NONE ? nullptr : (const half_t *)bias;
    a.residual = (const half_t *)residual;
    a.M = (int)T; a.N = (int)F; a.K = (int)K; a.NB = (int)F;
    a.ldY = ldY; a.ldA = ldX; a.ldB = ldW; a.sY = sY; a.sA = sX; a.sB = sW; a.sBias = sBias; a.dRes = 0;
    a.bias_mode = bias_mode; a.epi = epi; a.out_f32 = out_dtype == MI_F32;
    a.tiles_m = a.tiles_n = a.group_m = 1; a.vec_store = 0;
    a.cv = ConvGather{};
    a.ag = NhwcGather{};
    a.ln_gamma = a.ln_beta = nullptr; a.ln_eps = 0.0f; a.ln_on = 0; a.div_k8 = K >= 8 ? recip_of(K / 8) : 0;
    a.lnout = nullptr; a.lnout_gamma = a.lnout_beta = nullptr; a.lnout_eps = 0.0f; a.clamp = 0.0f;
    a.clk = nullptr; a.phase = nullptr; a.phase_wgs = 0;
    a.sk_S = 0; a.sk_tpx = 0; a.sk_part = nullptr; a.sk_flags = nullptr; a.sk_epoch = 0;
    a.sk_spin = 0; a.sk_pub_xor = a.sk_xcc_xor = 0; a.status = nullptr;
    a.lnf_stats = a.lnf_colsum = a.lnf_biasp = nullptr; a.lnf_svec = 0; a.lnf_nseg = 0; a.lnf_eps = 0.0f; a.stats_out = nullptr; a.stats_nseg = 0;
    return MI_OK;
}

// Internal status: the split-K epilogue has also written a.lnout (the caller must not run the norm again).
constexpr int MI_LNOUT_DONE = -1;

bool lnout_rowwise_ok(const GemmArgs &a) {
    return !a.out_f32 && a.N % 8 == 0 && a.N <= 4096 && a.ldY % 8 == 0 && aligned_to(a.Y, 16) && aligned_to(a.lnout, 16) &&
           (!a.residual || aligned_to(a.residual, 16)) && (!a.lnout_gamma || aligned_to(a.lnout_gamma, 16)) &&
           (!a.lnout_beta || aligned_to(a.lnout_beta, 16));
}

int run_gemm(GemmArgs a, bool b_kn, int64_t nbatch, void *ws, size_t ws_bytes, hipStream_t st, int force_path) {
    if (!g_ready) return MI_ERROR_DEVICE;
    if (a.M == 0 || a.N == 0 || nbatch == 0) return MI_OK;
    int path = force_path ? force_path : gemm_path(a, b_kn, nbatch);
    if (path == MI_GEMM_DECLINE) return MI_DECLINE_EXTENT;
    if (path == MI_GEMM_SKINNY) return mi_skinny_launch(a, b_kn, ws, ws_bytes, st);
    if (path == MI_GEMM_MFMA) {
        if (!mfma_addressable(a, b_kn)) return MI_DECLINE_OPERANDS;
        // Split K over workgroups when the output alone cannot fill the chip: each K-slice is one plane
        // of a batched launch (plane strides: A advances along k, Y one fp32 M x N plane in ws), and a
        // second small kernel sums the planes and applies bias, activation and residual.
        const bool pipe = a.K > 64, whole = pipe && a.K % 64 == 0;
        if (a.ag.x && !whole) return MI_DECLINE_EXTENT;      // only the pipelined kernel gathers
        TilePlan tp = {4, 1, false, 0.0};
        // A folded norm on the way in or row statistics on the way out live in the tiled kernels' own store: those calls
        // need the pipelined kernels, 16-byte rows, and K-slices only in the form that ends in that store (the in-launch
        // exchange), never planes.
        const bool in_store = a.lnf_stats || a.stats_out;
        if (in_store) {
            const bool rows16 = !a.out_f32 ? (a.N % 8 == 0 && a.ldY % 8 == 0 && a.sY % 8 == 0 && aligned_to(a.Y, 16) && (!a.residual || aligned_to(a.residual, 16)))
                                           : (a.N % 4 == 0 && a.ldY % 4 == 0 && a.sY % 4 == 0 && aligned_to(a.Y, 16));
            if (!whole || a.ag.x || !rows16 || (a.stats_out && a.out_f32)) return MI_DECLINE_EXTENT;
        }
        const bool deep = !a.ag.x, lnf = a.lnf_stats;
        if (pipe) {
            tp = plan_tiles(a.M, a.N, a.K, nbatch, !lnf, false, deep, lnf);
            if (tp.split > 1 && !(ws && aligned_to(ws, 256) && ws_bytes >= plan_workspace_bytes(tp, a.M, a.N)))
                tp = plan_tiles(a.M, a.N, a.K, nbatch, false, false, deep, lnf);
            if (in_store && tp.split > 1 && !(tp.peer && sk_usable())) tp = plan_tiles(a.M, a.N, a.K, nbatch, false, false, deep, lnf);
        }
        int split = tp.split;
        if (split > 1 && tp.peer && ws && aligned_to(ws, 256) && ws_bytes >= plan_workspace_bytes(tp, a.M, a.N)) {
            const int rc = launch_w4_peer(a, b_kn, split, ws, st);
            if (rc != MI_DECLINE_EXTENT) return rc;     // declined (a gathered operand, a device that failed the probe): planes
            if (in_store) { tp = plan_tiles(a.M, a.N, a.K, nbatch, false, false, deep, lnf); split = 1; }
        }
        if (split > 1 && ws && aligned_to(ws, 256) && ws_bytes >= (size_t)split * a.M * a.N * sizeof(float)) {
            GemmArgs s1 = a;
            s1.Y = ws; s1.out_f32 = 1; s1.bias = nullptr; s1.bias_mode = MI_BIAS_NONE; s1.epi = MI_EPI_NONE; s1.residual = nullptr; s1.clamp = 0.0f;
            s1.ldY = a.N; s1.sY = (long)a.M * a.N;
            s1.K = a.K / split;
            s1.sA = s1.K; s1.sB = b_kn ? (long)s1.K * a.ldB : s1.K; s1.sBias = 0;
            s1.ag.split = 1;
            int rc = launch_tile(tp.tile, s1, b_kn, split, st);
            if (rc != MI_OK) return rc;
            GemmArgs s2 = a;
            s2.vec_store = !a.out_f32 && a.ldY % 4 == 0 && aligned_to(a.Y, 8);
            const float *planes = reinterpret_cast<const float *>(ws);
            if (a.lnout && lnout_rowwise_ok(a)) {
                // the norm of the finished rows rides in the pass that sums the planes: one wave per row
                dim3 grid((unsigned)ceil_div(a.M, 4));
                if (a.N <= 512)       hipLaunchKernelGGL(splitk_epilogue_ln_kernel<1>, grid, dim3(256), 0, st, s2, planes, split);
                else if (a.N <= 1024) hipLaunchKernelGGL(splitk_epilogue_ln_kernel<2>, grid, dim3(256), 0, st, s2, planes, split);
                else if (a.N <= 2048) hipLaunchKernelGGL(splitk_epilogue_ln_kernel<4>, grid, dim3(256), 0, st, s2, planes, split);
                else                  hipLaunchKernelGGL(splitk_epilogue_ln_kernel<8>, grid, dim3(256), 0, st, s2, planes, split);
                return hipGetLastError() == hipSuccess ? MI_LNOUT_DONE : MI_ERROR_LAUNCH;
            }
            const long quads = ((long)a.M * a.N) / 4;
            hipLaunchKernelGGL(splitk_epilogue_kernel, dim3((unsigned)ceil_div(quads, 256)), dim3(256), 0, st, s2, planes, split);
            return hipGetLastError() == hipSuccess ? MI_OK : MI_ERROR_LAUNCH;
        }
        // A GELU store is some fifteen vector instructions a value, so narrower tiles can be the faster ones for it (1500 x 384 ->
        // 1536: 9.1 us on 128 x 128, 8.0 on 64 x 64).  The choice is among the tiles that sum K in the same order, or stays with one that
        // has its own: the bits are the ones without a GELU.
        if (pipe && split == 1 && !own_order(tp.tile, a.K) && (a.epi == MI_EPI_GELU_ERF || a.epi == MI_EPI_GELU_TANH))
            tp = plan_tiles(a.M, a.N, a.K, nbatch, false, true, deep, lnf);
        if (pipe) return launch_tile(settled_tile(tp.tile, a, nbatch), a, b_kn, nbatch, st);
        return mi_any_launch(a, b_kn, true, nbatch, st);         // a single tile deep
    }
    return mi_any_launch(a, b_kn, false, nbatch, st);
}

}  // namespace

bool mi_ready() { return g_ready; }
int mi_num_cus() { return tl_plan_cus > 0 ? tl_plan_cus : g_cus; }
bool mi_plan_mfma() { return tl_plan_mfma; }
void mi_plan_caps_begin(const int64_t *caps) {
    if (!caps) return;
    tl_plan_mfma = caps[0] != 0;
    tl_plan_cus = caps[5] > 0 ? (int)(caps[5] > 65536 ? 65536 : caps[5]) : 1;
}
void mi_plan_caps_end() { tl_plan_cus = 0; tl_plan_mfma = true; }
bool mi_xcd_round_robin() { return sk_usable(); }

// Split-K planes of a GEMM issued through mi_internal_gemm.
size_t mi_internal_gemm_workspace(int64_t T, int64_t K, int64_t F, int64_t nbatch) {
    if (T <= 8) return mi_gemm_f16_workspace(T, K, F, MI_W_KF, nbatch);      // decode-sized: the [K][F] kernel's planes
    if (nbatch > 1 || K % 64 || K < 128) return 0;
    return planned_workspace(T, F, K);
}

// A patch matrix is gathered by two kernels: 64 x 64 tiles, and 32 x 32 ones with K split over their waves where they are at most one
// workgroup a CU (as many as their estimate was fitted to): 43 such convolutions 0.62 to 0.96 of the ring's time.
static bool patches_deep(int64_t T, int64_t K, int64_t F, int64_t nbatch) {
    return ceil_div(T, 32) * ceil_div(F, 32) * nbatch <= std::min(DEEP_WGS, (int64_t)mi_num_cus()) &&
           tile_cost_us(T, F, K, nbatch, DEEP_TILE, 1) < tile_cost_us(T, F, K, nbatch, RING_TILE, 1);
}
double mi_internal_patch_gemm_us(int64_t T, int64_t K, int64_t F, int64_t nbatch) { return tile_cost_us(T, F, K, nbatch, patches_deep(T, K, F, nbatch) ? DEEP_TILE : RING_TILE, 1); }
int mi_internal_patch_kernel(int64_t T, int64_t K, int64_t F, int64_t nbatch) {
    if (patches_deep(T, K, F, nbatch)) return MI_GEMM_KERNEL_DEEP;
    return ceil_div(T, 64) * ceil_div(F, 64) * nbatch <= mi_num_cus() ? MI_GEMM_KERNEL_RING : MI_GEMM_KERNEL_RING_SHALLOW;
}
double mi_deep_us(int64_t T, int64_t K, int64_t F) {
    return ceil_div(T, 32) * ceil_div(F, 32) <= std::min(DEEP_WGS, (int64_t)mi_num_cus()) ? tile_cost_us(T, F, K, 1, DEEP_TILE, 1) : 1e30;
}
double mi_internal_gemm_us(int64_t T, int64_t K, int64_t F, int64_t nbatch) { return plan_tiles(T, F, K, nbatch, nbatch == 1).us; }

// Internal entry used by the convolution path (conv.hip): Y[M x N] = A . B with
// every GemmArgs field meaningful.
int mi_internal_gemm(void *Y, const void *A, const void *B, const void *bias, int M, int N, int NB, int K,
                     long ldY, long ldA, long ldB, int b_kn, int bias_mode, int epi, int out_f32,
                     long nbatch, long sY, long sA, long sB, void *ws, size_t ws_bytes, hipStream_t st,
                     const ConvGather *gather, const NhwcGather *agather, const void *residual, long dres) {
    GemmArgs a;
    a.cv = ConvGather{};
    a.ag = NhwcGather{};
    a.ln_gamma = a.ln_beta = nullptr; a.ln_eps = 0.0f; a.ln_on = 0; a.div_k8 = K >= 8 ? recip_of(K / 8) : 0;
    a.lnout = nullptr; a.lnout_gamma = a.lnout_beta = nullptr; a.lnout_eps = 0.0f; a.clamp = 0.0f;
    a.clk = nullptr; a.phase = nullptr; a.phase_wgs = 0;
    a.sk_S = 0; a.sk_tpx = 0; a.sk_part = nullptr; a.sk_flags = nullptr; a.sk_epoch = 0;
    a.sk_spin = 0; a.sk_pub_xor = a.sk_xcc_xor = 0; a.status = nullptr;
    a.lnf_stats = a.lnf_colsum = a.lnf_biasp = nullptr; a.lnf_svec = 0; a.lnf_nseg = 0; a.lnf_eps = 0.0f; a.stats_out = nullptr; a.stats_nseg = 0;
    a.Y = Y; a.A = (const half_t *)A; a.B = (const half_t *)B; a.bias = (const half_t *)bias; a.residual = out_f32 ? nullptr : (const half_t *)residual;
    a.M = M; a.N = N; a.NB = NB; a.K = K; a.ldY = ldY; a.ldA = ldA; a.ldB = ldB; a.sY = sY; a.sA = sA; a.sB = sB; a.sBias = 0; a.dRes = dres;
    a.bias_mode = bias ? bias_mode : MI_BIAS_NONE; a.epi = epi; a.out_f32 = out_f32;
    a.tiles_m = a.tiles_n = a.group_m = 1; a.vec_store = 0;
    if (gather) a.cv = *gather;
    if (agather) a.ag = *agather;
    const bool addr = mfma_addressable(a, b_kn != 0);
    if ((gather || agather) && !addr) return MI_DECLINE_OPERANDS;
    if (gather) {
        if (!g_ready) return MI_ERROR_DEVICE;
        return patches_deep(M, K, N, nbatch) ? mi_deep_launch(a, true, false, nbatch, st) : mi_ring_launch(a, false, nbatch, st);
    }
    int path = addr ? MI_GEMM_MFMA : MI_GEMM_SCALAR;
    return run_gemm(a, b_kn != 0, nbatch, ws, ws_bytes, st, path);
}

extern "C" {

int mi_version(void) { return MI355DNN_VERSION; }

int mi_init(void) {
    if (g_ready) return MI_OK;
    int dev = 0;
    if (hipGetDevice(&dev) != hipSuccess) return MI_ERROR_DEVICE;
    hipDeviceProp_t prop;
    if (hipGetDeviceProperties(&prop, dev) != hipSuccess) return MI_ERROR_DEVICE;
    if (__builtin_strncmp(prop.gcnArchName, "gfx950", 6) != 0) return MI_ERROR_DEVICE;
    g_cus = prop.multiProcessorCount > 0 ? prop.multiProcessorCount : 256;
    int bad = 0;
    bad |= raise_lds(gemm_w4_kernel<128, 256, 1, 4, true>, w4_lds_bytes<128, 256>());
    bad |= raise_lds(gemm_w4_kernel<128, 256, 1, 4, false>, w4_lds_bytes<128, 256>());
    bad |= raise_lds(gemm_w4_kernel<192, 128, 2, 2, true>, w4_lds_bytes<192, 128>());
    bad |= raise_lds(gemm_w4_kernel<192, 128, 2, 2, false>, w4_lds_bytes<192, 128>());
    bad |= raise_lds(gemm_w4_kernel<128, 128, 2, 2, true, true>, w4_lds_bytes<128, 128>());
    bad |= raise_lds(gemm_w4_kernel<128, 128, 2, 2, false, true>, w4_lds_bytes<128, 128>());
    bad |= mi_skinny_init() | mi_pipe_init() | mi_ring_init() | mi_deep_init() | mi_any_init() | mi_conv_tile_init();
    bad |= mi_sdpa_init();
    bad |= scratch_of_current_device() == nullptr;
    sk_probe_current_device();      // a device that fails the probe only loses that path
    if (bad) return MI_ERROR_DEVICE;
    g_ready = true;
    return MI_OK;
}

int mi_set_phase_probe(void *dev_u64, int64_t workgroups) {
    if (workgroups < 0 || workgroups > (1 << 20) || (dev_u64 && !aligned_to(dev_u64, 8))) return MI_DECLINE_OPERANDS;
    g_phase_probe = reinterpret_cast<unsigned long long *>(dev_u64);
    g_phase_wgs = dev_u64 ? (int)workgroups : 0;
    return MI_OK;
}

int mi_set_clock_probe(void *dev_u64x4) {
    if (dev_u64x4 && !aligned_to(dev_u64x4, 8)) return MI_DECLINE_OPERANDS;
    g_clock_probe = reinterpret_cast<unsigned long long *>(dev_u64x4);
    return MI_OK;
}

int mi_device_status(int reset) {
    int dev = -1;
    if (hipGetDevice(&dev) != hipSuccess || dev < 0 || dev >= MAX_DEVICES || !g_status_ptr[dev]) return -1;
    if (hipDeviceSynchronize() != hipSuccess) return -1;
    unsigned word = 0;
    if (hipMemcpy(&word, g_status_ptr[dev], sizeof(word), hipMemcpyDeviceToHost) != hipSuccess) return -1;
    if (reset) {
        // a wave that gave up released nothing: zero every bank of flags and counters along with the word
        bool ok = hipMemset(g_status_ptr[dev], 0, sizeof(unsigned)) == hipSuccess;
        if (g_sk_flags_ptr[dev]) ok = ok && hipMemset(g_sk_flags_ptr[dev], 0, sizeof(unsigned) * 2 * SK_WORDS) == hipSuccess;
        if (!ok || hipDeviceSynchronize() != hipSuccess) return -1;
    }
    return (int)(word & 0x7fffffffu);
}

int mi_set_in_launch_exchange(int enabled) {
    g_sk_enabled.store(enabled != 0);
    return MI_OK;
}

int mi_test_exchange_faults(int spin_limit, unsigned publish_xor, unsigned xcc_xor) {
    g_sk_spin = spin_limit > 0 ? spin_limit : SK_SPIN_DEFAULT;
    g_sk_pub_xor = publish_xor & sk::EPOCH_MASK;
    g_sk_xcc_xor = xcc_xor & 15u;
    return MI_OK;
}

int mi_device_caps(int64_t out[6]) {
    if (!out) return MI_DECLINE_OPERANDS;
    int dev = 0;
    hipDeviceProp_t prop;
    if (hipGetDevice(&dev) != hipSuccess || hipGetDeviceProperties(&prop, dev) != hipSuccess) return MI_ERROR_DEVICE;
    out[0] = __builtin_strncmp(prop.gcnArchName, "gfx950", 6) == 0;
    out[1] = 16;
    out[2] = prop.warpSize;
    out[3] = (int64_t)prop.maxSharedMemoryPerMultiProcessor;
    out[4] = prop.maxThreadsPerBlock;
    out[5] = prop.multiProcessorCount;
    return MI_OK;
}

size_t mi_gemm_f16_workspace(int64_t T, int64_t K, int64_t F, int w_layout, int64_t nbatch) {
    if (T < 1 || nbatch > 1) return 0;
    if (T > 8) {
        if (K % 64 || K < 128) return 0;
        // Room for the exchange wherever it can run on a K of some length, whichever tile the estimate prefers: buffers and
        // recorded plans keep their sizes when its constants move.
        const size_t need = planned_workspace(T, F, K);
        const TileModel &t = TILE_MODELS[SK_TILE];
        const size_t peer = K >= 2048 && sk_fits(T, F, K, t.bm, t.bn, 2) ? round_up(sk_workspace_bytes(T, F, t.bm, t.bn, 2), 256) : 0;
        return need > peer ? need : peer;
    }
    if (w_layout != MI_W_KF) return 0;      // the [F][K] skinny kernel finishes its outputs itself
    return round_up((size_t)mi_skinny_splits(K, F) * T * F * sizeof(float), 256);
}

int mi_gemm_f16_plan(const void *Y, const void *X, const void *W,
                     int64_t T, int64_t K, int64_t F, int64_t ldY, int64_t ldX, int64_t ldW,
                     int w_layout, int out_dtype, int64_t nbatch, int64_t sY, int64_t sX, int64_t sW) {
    GemmArgs a;
    int rc = fill_args(a, const_cast<void *>(Y), X, W, nullptr, nullptr, T, K, F, ldY, ldX, ldW, w_layout, MI_BIAS_NONE,
                       MI_EPI_NONE, out_dtype, sY, sX, sW);
    if (rc != MI_OK) return MI_GEMM_DECLINE;
    return gemm_path(a, w_layout == MI_W_KF, nbatch < 1 ? 1 : nbatch);
}

int mi_gemm_f16_plan_caps(const int64_t caps[6], const void *Y, const void *X, const void *W,
                          int64_t T, int64_t K, int64_t F, int64_t ldY, int64_t ldX, int64_t ldW,
                          int w_layout, int out_dtype, int64_t nbatch, int64_t sY, int64_t sX, int64_t sW, int *ksplit_out) {
    mi_plan_caps_begin(caps);
    const int path = mi_gemm_f16_plan(Y, X, W, T, K, F, ldY, ldX, ldW, w_layout, out_dtype, nbatch, sY, sX, sW);
    if (ksplit_out) {
        *ksplit_out = 1;
        if (path == MI_GEMM_MFMA && K % 64 == 0 && K >= 128) *ksplit_out = plan_tiles(T, F, K, nbatch < 1 ? 1 : nbatch, true).split;
        if (path == MI_GEMM_SKINNY && w_layout == MI_W_KF) *ksplit_out = mi_skinny_slices(T, K, F, ldX, ldW);
    }
    mi_plan_caps_end();
    return path;
}

int mi_gemm_f16_kernel(int64_t T, int64_t K, int64_t F, int64_t nbatch, int epi, int folded_norm, int *ksplit_out) {
    if (ksplit_out) *ksplit_out = 1;
    if (T <= 8 || K < 8 || K % 8 || F < 8 || F % 8 || nbatch < 1 || T > INT32_MAX || K > INT32_MAX || F > INT32_MAX) return MI_GEMM_KERNEL_NONE;
    if (K <= 64) return MI_GEMM_KERNEL_ONE_TILE;
    const bool lnf = folded_norm != 0;
    TilePlan tp = plan_tiles(T, F, K, nbatch, !lnf, false, true, lnf);
    if (tp.split == 1 && !own_order(tp.tile, K) && (epi == MI_EPI_GELU_ERF || epi == MI_EPI_GELU_TANH)) tp = plan_tiles(T, F, K, nbatch, false, true, true, lnf);
    if (ksplit_out) *ksplit_out = tp.split;
    if (tp.peer) return MI_GEMM_KERNEL_EXCHANGE;
    if (tp.split == 1 && !lnf) {
        GemmArgs a = {};
        a.M = (int)T; a.N = (int)F; a.K = (int)K; a.epi = epi;
        tp.tile = settled_tile(tp.tile, a, nbatch);
    }
    switch (tp.tile) {
        case 0: case 1: return MI_GEMM_KERNEL_WIDE;
        case RING_TILE: return ceil_div(T, 64) * ceil_div(F, 64) * nbatch * tp.split <= mi_num_cus() ? MI_GEMM_KERNEL_RING : MI_GEMM_KERNEL_RING_SHALLOW;
        case DEEP_TILE: return MI_GEMM_KERNEL_DEEP;
        case DEEP_SERIAL_TILE: return MI_GEMM_KERNEL_DEEP_SERIAL;
        default: return MI_GEMM_KERNEL_STAGED;
    }
}

int mi_gemm_f16_batched(void *Y, const void *X, const void *W, const void *bias, const void *residual,
                        int64_t T, int64_t K, int64_t F, int64_t ldY, int64_t ldX, int64_t ldW,
                        int w_layout, int bias_mode, int epi, int out_dtype,
                        int64_t nbatch, int64_t sY, int64_t sX, int64_t sW, int64_t sBias,
                        void *ws, size_t ws_bytes, void *stream) {
    GemmArgs a;
    int rc = fill_args(a, Y, X, W, bias, residual, T, K, F, ldY, ldX, ldW, w_layout, bias_mode, epi, out_dtype, sY, sX, sW, sBias);
    if (rc != MI_OK) return rc;
    if (nbatch < 0 || nbatch > 65535) return MI_DECLINE_EXTENT;
    if (K == 0) return MI_DECLINE_EXTENT;
    return run_gemm(a, w_layout == MI_W_KF, nbatch, ws, ws_bytes, (hipStream_t)stream, 0);
}

int mi_gemm_f16(void *Y, const void *X, const void *W, const void *bias, const void *residual,
                int64_t T, int64_t K, int64_t F, int64_t ldY, int64_t ldX, int64_t ldW,
                int w_layout, int bias_mode, int epi, int out_dtype,
                void *ws, size_t ws_bytes, void *stream) {
    return mi_gemm_f16_batched(Y, X, W, bias, residual, T, K, F, ldY, ldX, ldW, w_layout, bias_mode, epi, out_dtype,
                               1, 0, 0, 0, 0, ws, ws_bytes, stream);
}

int mi_gemm_ln_f16(void *Y, void *H, const void *X, const void *W, const void *bias, const void *residual,
                   const void *gamma, const void *beta, float eps,
                   int64_t T, int64_t K, int64_t F, int64_t ldX, int64_t ldW,
                   int w_layout, int bias_mode, int epi, void *ws, size_t ws_bytes, void *stream) {
    if (!H) return MI_DECLINE_OPERANDS;
    GemmArgs a;
    int rc = fill_args(a, Y, X, W, bias, residual, T, K, F, F, ldX, ldW, w_layout, bias_mode, epi, MI_F16, 0, 0, 0);
    if (rc != MI_OK) return rc;
    if (!g_ready) return MI_ERROR_DEVICE;
    a.lnout = (half_t *)H; a.lnout_gamma = (const half_t *)gamma; a.lnout_beta = (const half_t *)beta; a.lnout_eps = eps;
    rc = run_gemm(a, w_layout == MI_W_KF, 1, ws, ws_bytes, (hipStream_t)stream, 0);
    if (rc == MI_LNOUT_DONE) return MI_OK;
    if (rc != MI_OK) return rc;
    return mi_layernorm_f16(H, nullptr, nullptr, Y, gamma, beta, F, T, eps, stream);      // rows of Y are dense: ldY = F
}

int mi_gemm_clamp_ln_f16(void *Y, void *H, const void *X, const void *W, const void *bias, const void *residual,
                         const void *gamma, const void *beta, float eps, float clamp,
                         int64_t T, int64_t K, int64_t F, int64_t ldX, int64_t ldW,
                         int w_layout, int bias_mode, int epi, void *ws, size_t ws_bytes, void *stream) {
    if (is_nan_arg(clamp) || clamp <= 0.0f) return MI_DECLINE_OPERANDS;
    GemmArgs a;
    int rc = fill_args(a, Y, X, W, bias, residual, T, K, F, F, ldX, ldW, w_layout, bias_mode, epi, MI_F16, 0, 0, 0);
    if (rc != MI_OK) return rc;
    if (!g_ready) return MI_ERROR_DEVICE;
    if (T == 0 || F == 0) return MI_OK;
    const bool b_kn = w_layout == MI_W_KF;
    // the tiled kernels and the plane sums clamp in their stores; the decode-sized and scalar kernels do not: there the
    // clamp is a pass of its own over Y
    const bool in_store = gemm_path(a, b_kn, 1) == MI_GEMM_MFMA;
    if (in_store) a.clamp = clamp;
    if (H) { a.lnout = (half_t *)H; a.lnout_gamma = (const half_t *)gamma; a.lnout_beta = (const half_t *)beta; a.lnout_eps = eps; }
    if (!in_store) a.lnout = nullptr;
    rc = run_gemm(a, b_kn, 1, ws, ws_bytes, (hipStream_t)stream, 0);
    if (rc == MI_LNOUT_DONE) return MI_OK;
    if (rc != MI_OK) return rc;
    if (!in_store) {
        rc = mi_clamp_f16(Y, Y, -clamp, clamp, T * F, stream);
        if (rc != MI_OK) return rc;
    }
    return H ? mi_layernorm_f16(H, nullptr, nullptr, Y, gamma, beta, F, T, eps, stream) : MI_OK;
}

int mi_gemm_rowstats_f16(void *Y, float *stats, const void *X, const void *W, const void *bias, const void *residual, float clamp,
                         int64_t T, int64_t K, int64_t F, int64_t ldX, int64_t ldW,
                         int w_layout, int bias_mode, int epi, void *ws, size_t ws_bytes, void *stream) {
    if (!stats || !aligned_to(stats, 8) || is_nan_arg(clamp)) return MI_DECLINE_OPERANDS;
    GemmArgs a;
    int rc = fill_args(a, Y, X, W, bias, residual, T, K, F, F, ldX, ldW, w_layout, bias_mode, epi, MI_F16, 0, 0, 0);
    if (rc != MI_OK) return rc;
    if (!g_ready) return MI_ERROR_DEVICE;
    if (T == 0 || F == 0) return MI_OK;
    if (gemm_path(a, w_layout == MI_W_KF, 1) != MI_GEMM_MFMA) return MI_DECLINE_EXTENT;
    a.stats_out = stats; a.stats_nseg = (int)ceil_div(F, 32);
    if (clamp > 0.0f) a.clamp = clamp;
    return run_gemm(a, w_layout == MI_W_KF, 1, ws, ws_bytes, (hipStream_t)stream, 0);
}

int mi_lnfold_gemm_f16(void *Y, float *stats_out, const void *X, const float *stats_in, float eps,
                       const void *Wp, const float *colsum, const float *biasp, const void *residual, float clamp,
                       int64_t T, int64_t K, int64_t F, int64_t ldY, int64_t ldX, int64_t ldW,
                       int w_layout, int epi, int out_dtype,
                       int64_t nbatch, int64_t sY, int64_t sW, int64_t sVec, void *ws, size_t ws_bytes, void *stream) {
    if (!stats_in || !colsum || !biasp || !aligned_to(stats_in, 8) || !aligned_to(colsum, 16) || !aligned_to(biasp, 16) || sVec % 4) return MI_DECLINE_OPERANDS;
    if (is_nan_arg(eps) || is_nan_arg(clamp) || (stats_out && !aligned_to(stats_out, 8))) return MI_DECLINE_OPERANDS;
    if (nbatch < 1 || nbatch > 65535 || (stats_out && (nbatch != 1 || ldY != F || out_dtype != MI_F16))) return MI_DECLINE_EXTENT;
    GemmArgs a;
    int rc = fill_args(a, Y, X, Wp, nullptr, residual, T, K, F, ldY, ldX, ldW, w_layout, MI_BIAS_NONE, epi, out_dtype, sY, 0, sW);
    if (rc != MI_OK) return rc;
    if (!g_ready) return MI_ERROR_DEVICE;
    if (T == 0 || F == 0) return MI_OK;
    if (T <= 8 || !mfma_addressable(a, w_layout == MI_W_KF)) return MI_DECLINE_EXTENT;      // decode-sized rows: mi_ln_gemv_f16
    a.lnf_stats = stats_in; a.lnf_nseg = (int)ceil_div(K, 32); a.lnf_eps = eps;
    a.lnf_colsum = colsum; a.lnf_biasp = biasp; a.lnf_svec = sVec;
    if (stats_out) { a.stats_out = stats_out; a.stats_nseg = (int)ceil_div(F, 32); }
    if (clamp > 0.0f) a.clamp = clamp;
    return run_gemm(a, w_layout == MI_W_KF, nbatch, ws, ws_bytes, (hipStream_t)stream, MI_GEMM_MFMA);
}

// mi_gemm_f16 for callers that cannot allocate: the split-K / decode planes go to `scratch`, a file-scope
// device array, reached through the per-device address that hipGetSymbolAddress returns (the array's name is only a
// host-side stand-in).  The planes are written in full before they are summed, so nothing needs clearing between calls.
int mi_gemm_f16_noalloc(void *Y, const void *X, const void *W, const void *bias, const void *residual,
                        int64_t T, int64_t K, int64_t F, int64_t ldY, int64_t ldX, int64_t ldW,
                        int w_layout, int bias_mode, int epi, int out_dtype, void *stream) {
    if (!g_ready) return MI_ERROR_DEVICE;
    const size_t need = mi_gemm_f16_workspace(T, K, F, w_layout, 1);
    if (need > (size_t)MI_NOALLOC_SCRATCH_BYTES) return MI_DECLINE_SCRATCH_LIMIT;
    void *planes = nullptr;
    if (need) {
        planes = scratch_of_current_device();
        if (!planes) return MI_ERROR_DEVICE;
    }
    return mi_gemm_f16(Y, X, W, bias, residual, T, K, F, ldY, ldX, ldW, w_layout, bias_mode, epi, out_dtype,
                       planes, need ? (size_t)MI_NOALLOC_SCRATCH_BYTES : 0, stream);
}

int mi_gemv_f16(void *Y, const void *X, const void *W, const void *bias, const void *residual,
                int64_t T, int64_t K, int64_t F, int64_t ldY, int64_t ldX, int64_t ldW,
                int w_layout, int bias_mode, int epi, int out_dtype,
                void *ws, size_t ws_bytes, void *stream) {
    GemmArgs a;
    int rc = fill_args(a, Y, X, W, bias, residual, T, K, F, ldY, ldX, ldW, w_layout, bias_mode, epi, out_dtype, 0, 0, 0);
    if (rc != MI_OK) return rc;
    if (!g_ready) return MI_ERROR_DEVICE;
    if (T < 1 || T > 8) return MI_DECLINE_EXTENT;
    if (!mfma_addressable(a, w_layout == MI_W_KF)) return MI_DECLINE_OPERANDS;
    return mi_skinny_launch(a, w_layout == MI_W_KF, ws, ws_bytes, (hipStream_t)stream);
}

int mi_ln_gemm_f16(void *Y, const void *X, const void *gamma, const void *beta, float eps,
                   const void *W, const void *bias, const void *residual,
                   int64_t T, int64_t K, int64_t F, int64_t ldY, int64_t ldX, int64_t ldW,
                   int w_layout, int bias_mode, int epi, int out_dtype,
                   void *ws, size_t ws_bytes, void *stream) {
    if (T >= 1 && T <= 8)
        return mi_ln_gemv_f16(Y, X, gamma, beta, eps, W, bias, residual, T, K, F, ldY, ldX, ldW, w_layout, bias_mode, epi,
                              out_dtype, ws, ws_bytes, stream);
    GemmArgs a;
    int rc = fill_args(a, Y, X, W, bias, residual, T, K, F, ldY, ldX, ldW, w_layout, bias_mode, epi, out_dtype, 0, 0, 0);
    if (rc != MI_OK) return rc;
    if (!g_ready) return MI_ERROR_DEVICE;
    if (T == 0 || F == 0) return MI_OK;
    const bool b_kn = w_layout == MI_W_KF;
    if (!mfma_addressable(a, b_kn)) return MI_DECLINE_OPERANDS;
    if ((gamma && !aligned_to(gamma, 16)) || (beta && !aligned_to(beta, 16))) return MI_DECLINE_OPERANDS;
    if (K < 128 || K % 64 || K > MI_LNA_KMAX) return MI_DECLINE_EXTENT;      // the caller runs the two ops
    // a shape whose plain GEMM would split K sums in another order: keep the promise of identical bits, decline
    if (plan_tiles(T, F, K, 1, true).split != 1) return MI_DECLINE_EXTENT;
    a.ln_on = 1; a.ln_gamma = (const half_t *)gamma; a.ln_beta = (const half_t *)beta; a.ln_eps = eps;
    // 64-row tiles only (the normalised panel of a workgroup stays in LDS); which width, by the same estimate as
    // every other tiled launch
    const bool wide = tile_cost_us(T, F, K, 1, 3, 1) <= tile_cost_us(T, F, K, 1, 4, 1);
    return mi_pipe_launch_ln(wide, a, b_kn, (hipStream_t)stream);
}

int mi_ln_gemv_f16(void *Y, const void *X, const void *gamma, const void *beta, float eps,
                   const void *W, const void *bias, const void *residual,
                   int64_t T, int64_t K, int64_t F, int64_t ldY, int64_t ldX, int64_t ldW,
                   int w_layout, int bias_mode, int epi, int out_dtype,
                   void *ws, size_t ws_bytes, void *stream) {
    GemmArgs a;
    int rc = fill_args(a, Y, X, W, bias, residual, T, K, F, ldY, ldX, ldW, w_layout, bias_mode, epi, out_dtype, 0, 0, 0);
    if (rc != MI_OK) return rc;
    if (!g_ready) return MI_ERROR_DEVICE;
    if (T < 1 || T > 8) return MI_DECLINE_EXTENT;
    if (!mfma_addressable(a, w_layout == MI_W_KF)) return MI_DECLINE_OPERANDS;
    if ((gamma && !aligned_to(gamma, 16)) || (beta && !aligned_to(beta, 16))) return MI_DECLINE_OPERANDS;
    if (w_layout == MI_W_FK && (size_t)8 * K * sizeof(half_t) > SKINNY_FK_LDS_MAX) return MI_DECLINE_EXTENT;
    a.ln_on = 1; a.ln_gamma = (const half_t *)gamma; a.ln_beta = (const half_t *)beta; a.ln_eps = eps;
    return mi_skinny_launch(a, w_layout == MI_W_KF, ws, ws_bytes, (hipStream_t)stream);
}

}  // extern "C"
