#!/usr/bin/env python3
"""Benchmark of the dense-contraction hot path on one MI355X.

    python bench.py [--gpus 1] [--steps K] [--warmup W] [--detail/--no-detail] [--no-cpu]

A *step* is one Whisper-large-v3-turbo-shaped encoder block: batch 1, 1500
tokens, d_model 1280, 20 heads x 64, FFN 5120 with exact GELU, pre-LayerNorm, fp16 with fp32
accumulation, on synthetic seeded inputs already resident in HBM:

    LN -> q,k,v = h.Wq/Wk/Wv + b -> SDPA -> (.Wo + b) + x -> LN -> gelu(.W1 + b) -> (.W2 + b) + res

six kernel launches through the C ABI of libmi355dnn.so -- the q, k, v projections are one batched launch, and neither
layer norm is a pass of its own: both are folded into the linears that read them (mi_lnfold_gemm_f16, which runs on
the raw rows with per-row statistics left by the GEMM that wrote them, or by mi_rowstats_f16 for the block's input) -- captured once
as a HIP graph and replayed -- what the reference's runtime does with its own graphs (Lava.capture / replay) -- after
an untimed warm-up that runs until the step time has settled.  ``value`` is the block's algorithmic TFLOP/s (70.50 GFLOP
per block: 58.98 GEMM + 11.52 attention); ``ms_per_step`` is ms per encoder block; ``eager_ms_per_step`` the same steps
issued call by call.  ``roofline`` describes the dominant kernel -- the fp16 MFMA GEMM -- at whichever of its two largest
launches in the block takes longer, fc1 (1500x1280 -> 5120 + bias + GELU, BASELINE config 1's shape) or fc2
(1500x5120 -> 1280 + residual), each timed live with HIP events around the launch in at least 15 eager steps after the
timed loop; next to the fraction of the vendor's peak it carries what this box delivers with nothing in the way
(``peak_probe``: an MFMA-only kernel on a chip-filling grid and on config 1's own grid, a 256 MiB copy).
``cpu_baseline`` is the CPU oracle (a C port of the reference's KernelAbstractions-CPU forms) timed on this host on a
stated sample.  ``detail`` carries the other configs' kernels (config 1 GEMM in both weight layouts, config 4
attention and conv, config 3 shapes, config 5 decode linears and attention in GB/s), each timed
with HIP events over back-to-back launches on rotating buffer sets.

One JSON line is printed on stdout.
"""
from __future__ import annotations

import argparse
import ctypes as C
import json
import os
import sys
import time

ROOT = os.path.dirname(os.path.abspath(__file__))
if ROOT not in sys.path:
    sys.path.insert(0, ROOT)

PEAK_F16_TFLOPS = 2500.0       # MI355X dense fp16 MFMA, vendor figure
PEAK_HBM_GBS = 8000.0          # MI355X HBM3E, vendor figure

# HBM bytes per launch of the dominant kernel (fc1 GEMM) come from rocprofv3 --pmc FETCH_SIZE / WRITE_SIZE runs of
# `python bench.py --no-cpu --no-detail`, scaled by the same counters on a plain copy kernel of known size
# (--calibrate-copy).  The committed summary of those runs carries the figure on a line of its own; it is read from
# there, not restated here.
FC1_TRAFFIC_FILE = os.path.join("profiles", "fc1_gemm_hbm_traffic.txt")
MFMA_FLOP_PER_CLK_PER_CU = 4 * 1024     # four SIMDs, one v_mfma_f32_32x32x16_f16 (32 768 flop) per 32 cycles each


def fc_traffic_bytes(launch="fc1"):
    """``traffic_bytes_per_launch: N`` (fc1) or ``fc2_traffic_bytes_per_launch: N`` from the committed rocprofv3
    summary, or None if it is not there."""
    import re
    try:
        text = open(os.path.join(ROOT, FC1_TRAFFIC_FILE)).read()
    except OSError:
        return None
    key = "traffic_bytes_per_launch" if launch == "fc1" else "fc2_traffic_bytes_per_launch"
    m = re.search(r"^" + key + r":\s*(\d+)", text, re.M)
    return int(m.group(1)) if m else None


def peak_probe(lib, stream):
    """What this box delivers with nothing in the way, measured through the library's probe kernels: the matrix units
    on a chip-filling grid of nothing but MFMAs (random operands in registers), config 1's own grid -- 240 workgroups
    of eight waves, 20 steps of 16 MFMAs per wave, the GELU epilogue's arithmetic -- with every memory operation
    removed, and a 256 MiB device copy.  Medians of 15 event-timed samples after a warm-up of their own."""
    import torch
    seed = torch.randn(65536, dtype=torch.float16, device="cuda")
    sink = torch.zeros(512 * 4096, dtype=torch.float32, device="cuda")

    def timed(fn, reps):
        med, lo, hi = event_time(fn, reps)
        return med, lo

    def mfma(wgs, steps, gelu):
        rc = lib.mi_probe_mfma(sink.data_ptr(), seed.data_ptr(), wgs, steps, gelu, stream)
        if rc != 0:
            raise RuntimeError(f"mi_probe_mfma returned {rc}")
    # a grid of 16 rounds of one workgroup per CU, 100 steps each: 4096 x 8 waves x 1600 MFMAs of 32768 flop
    WG, STEPS = 4096, 100
    for _ in range(20):
        mfma(WG, STEPS, 0)
    t_fill, _ = timed(lambda: mfma(WG, STEPS, 0), 5)
    flop_fill = WG * 8 * STEPS * 16 * 32768.0
    t_c1, t_c1_min = timed(lambda: mfma(240, 20, 1), 20)
    t_c1_plain, _ = timed(lambda: mfma(240, 20, 0), 20)
    src = torch.empty(256 << 20, dtype=torch.uint8, device="cuda").random_(0, 255)
    dst = torch.empty_like(src)

    def copy():
        rc = lib.mi_probe_copy(dst.data_ptr(), src.data_ptr(), src.numel(), stream)
        if rc != 0:
            raise RuntimeError(f"mi_probe_copy returned {rc}")
    t_cp, _ = timed(copy, 5)
    # one phase boundary of a would-be multi-phase persistent kernel: every compute unit's workgroup at a grid barrier
    cus = torch.cuda.get_device_properties(0).multi_processor_count
    scratch = torch.zeros(576 + 8 * cus, dtype=torch.int32, device="cuda")
    ROUNDS = 200

    def barrier(payload):
        rc = lib.mi_probe_grid_barrier(scratch.data_ptr(), cus, ROUNDS, payload, stream)
        if rc != 0:
            raise RuntimeError(f"mi_probe_grid_barrier returned {rc}")
    t_bar, _ = timed(lambda: barrier(0), 5)
    t_bar_x, _ = timed(lambda: barrier(1), 5)
    gave_up = int(scratch[4].item())
    t_bar2, _ = timed(lambda: barrier(2), 5)
    t_bar2_x, _ = timed(lambda: barrier(3), 5)
    gave_up |= int(scratch[4].item())
    return {"grid_barrier_us": round(t_bar * 1e6 / ROUNDS, 2), "grid_barrier_with_exchange_us": round(t_bar_x * 1e6 / ROUNDS, 2),
            "grid_barrier_two_level_us": round(t_bar2 * 1e6 / ROUNDS, 2), "grid_barrier_two_level_with_exchange_us": round(t_bar2_x * 1e6 / ROUNDS, 2),
            "grid_barrier": f"{cus} workgroups, agent-scope atomic add + poll per round (two-level: eight groups with a counter and a release "
                            f"flag each); with exchange: 16 B published per workgroup "
                            f"before and all {16 * cus} B read back after; {ROUNDS} rounds per launch" + ("; SOME WAITS GAVE UP" if gave_up else ""),
            "mfma_only_tflops": round(flop_fill / t_fill / 1e12, 1),
            "mfma_only_frac_of_peak": round(flop_fill / t_fill / 1e12 / PEAK_F16_TFLOPS, 4),
            "mfma_only_grid": f"{WG} workgroups x 8 waves x {STEPS * 16} MFMAs (32x32x16 f16), no memory operations",
            "c1_no_memory_us": round(t_c1 * 1e6, 2), "c1_no_memory_us_min": round(t_c1_min * 1e6, 2),
            "c1_no_memory_no_gelu_us": round(t_c1_plain * 1e6, 2),
            "c1_no_memory_grid": "240 workgroups x 8 waves x 320 MFMAs + bias / rounding / erf-GELU on 64 values per lane, no memory operations",
            "hbm_copy_gbs": round(2.0 * src.numel() / t_cp / 1e9, 1), "hbm_copy_frac_of_peak": round(2.0 * src.numel() / t_cp / 1e9 / PEAK_HBM_GBS, 4),
            "hbm_copy": "256 MiB read + 256 MiB written by mi_probe_copy"}


def randn_f16(shape, seed, mean=0.0, std=1.0):
    """Seeded synthetic fp16 data (numpy's PCG64); the same host arrays feed the GPU step and the CPU baseline."""
    import numpy as np
    return (np.random.default_rng(seed).standard_normal(shape, dtype=np.float32) * std + mean).astype(np.float16)


def parse_args():
    ap = argparse.ArgumentParser()
    ap.add_argument("--gpus", type=int, default=1)
    ap.add_argument("--steps", type=int, default=200)
    ap.add_argument("--warmup", type=int, default=20)
    ap.add_argument("--detail", dest="detail", action="store_true", default=True)
    ap.add_argument("--no-detail", dest="detail", action="store_false")
    ap.add_argument("--no-cpu", dest="cpu", action="store_false", default=True)
    ap.add_argument("--only", default=None, metavar="SUBSTR",
                    help="run only the detail cases whose name contains SUBSTR (e.g. c4_attn, c1_linear) and print them; "
                         "for profiling one kernel with rocprofv3")
    ap.add_argument("--calibrate-copy", action="store_true",
                    help="also run a plain 256 MiB device copy (mi_probe_copy) three times, so that a rocprofv3 --pmc run "
                         "of this command holds a kernel of known HBM traffic to scale FETCH_SIZE / WRITE_SIZE by")
    ap.add_argument("--phase-stamps", action="store_true",
                    help="print where the waves of the four-wave GEMM kernel spend their clocks (mi_set_phase_probe) on config 1 "
                         "in both weight layouts and on the encoder block's q/k/v, fc1 and fc2 launches, and exit")
    return ap.parse_args()


def phase_stamps(lib, L, stream):
    """Shader clocks per matrix wave, averaged over all waves of ten launches: before the K loop (launch, addresses, the
    first operand tile's trip from memory), in the K loop (also per 64-deep tile, against the 1024 clocks -- 512 for the
    split-K instance's 64 x 64 wave tiles -- its MFMAs occupy the SIMD), issuing the store, waiting for it to drain."""
    import numpy as np
    import torch
    blk = EncoderBlock(lib, stream)
    blk.step()
    before, fc1, after = blk.calls_on(stream)
    T, D, FF = blk.T, blk.D, blk.FF
    p = lambda n: blk.d[n].data_ptr()
    wfk = blk.d["w1"].t().contiguous()

    def linear(layout, w, ldw):
        return Call(lib.mi_gemm_f16, p("f"), p("o"), w, p("b1"), None, T, D, FF, FF, D, ldw, layout, L.BIAS_COL, L.EPI["none"], L.F16,
                    blk._wsp, blk._ws_bytes, stream)
    cases = [("c1 1500x1280->5120 W[K][F] + bias", linear(L.W_KF, p("w1"), FF), 240, D // 64, 1024),
             ("c1 1500x1280->5120 W[F][K] + bias", linear(L.W_FK, wfk.data_ptr(), D), 240, D // 64, 1024),
             ("block q/k/v: LN1 folded, 3 planes, 192x128 tiles", before[1], 80, D // 64, 768),
             ("block fc1: LN2 folded + GELU, 128x256 tiles", fc1, 240, D // 64, 1024),
             ("block fc2: + residual, 128x128 tiles in two K-slices", after[0], 240, FF // 128, 512)]
    out = {}
    for name, call, wgs, nk, mfma in cases:
        for _ in range(30):
            call()
        buf = torch.zeros((wgs, 4, 4), dtype=torch.int64, device="cuda")
        if lib.mi_set_phase_probe(buf.data_ptr(), wgs) != 0:
            raise RuntimeError("mi_set_phase_probe")
        acc = np.zeros(4)
        for _ in range(10):
            buf.zero_()
            call()
            torch.cuda.synchronize()
            a = buf.cpu().numpy().astype(np.float64).reshape(-1, 4)
            acc += a[a.sum(1) > 0].mean(0)
        lib.mi_set_phase_probe(None, 0)
        m = acc / 10
        out[name] = {"before_loop": round(m[0]), "k_loop": round(m[1]), "k_loop_per_tile": round(m[1] / nk), "mfma_clocks_per_tile": mfma,
                     "store_issue": round(m[2]), "store_drain": round(m[3]), "total": round(m.sum())}
    return out


# ----------------------------------------------------------------------------- helpers

class Call:
    """A C-ABI call with its arguments converted once, so that issuing it costs one foreign call."""

    def __init__(self, fn, *args):
        self.fn = fn
        assert len(args) == len(fn.argtypes), (fn.__name__, len(args), len(fn.argtypes))
        self.args = tuple(a if (a is None or isinstance(a, (C._SimpleCData, C.Array))) else t(a)
                          for t, a in zip(fn.argtypes, args))

    def __call__(self):
        rc = self.fn(*self.args)
        if rc != 0:
            raise RuntimeError(f"{self.fn.__name__} returned status {rc}")


def dev(a):
    import numpy as np
    import torch
    return torch.from_numpy(np.ascontiguousarray(a)).cuda()


def event_time(fn, reps, samples=15):
    """Median seconds per call of fn() over `samples` groups of `reps` back-to-back launches."""
    import torch
    fn(); fn()
    torch.cuda.synchronize()
    ts = []
    for _ in range(samples):
        s = torch.cuda.Event(enable_timing=True)
        e = torch.cuda.Event(enable_timing=True)
        s.record()
        for i in range(reps):
            fn()
        e.record()
        e.synchronize()
        ts.append(s.elapsed_time(e) * 1e-3 / reps)
    ts.sort()
    return ts[len(ts) // 2], ts[0], ts[-1]


# ----------------------------------------------------------------------------- the encoder block

class EncoderBlock:
    T, D, H, E, FF = 1500, 1280, 20, 64, 5120
    FLOP_GEMM = 4 * (2 * 1500 * 1280 * 1280) + 2 * (2 * 1500 * 1280 * 5120)
    FLOP_ATTN = 4 * 1500 * 1500 * 64 * 20
    FLOP = FLOP_GEMM + FLOP_ATTN
    FC1_FLOP = 2 * 1500 * 1280 * 5120

    def __init__(self, lib, stream, seed=1000):
        import numpy as np
        import torch
        L = self.L = __import__("juliavision_amd")._lib
        T, D, H, E, FF = self.T, self.D, self.H, self.E, self.FF
        f16 = torch.float16
        self.host = {}
        h = self.host
        h["x"] = randn_f16((T, D), seed)
        h["wqkv"] = randn_f16((3, D, D), seed + 1, 0, 0.02)      # Wq, Wk, Wv, each [K][F]
        h["wo"] = randn_f16((D, D), seed + 4, 0, 0.02)
        h["w1"] = randn_f16((D, FF), seed + 5, 0, 0.02)
        h["w2"] = randn_f16((FF, D), seed + 6, 0, 0.02)
        h["bqkv"] = randn_f16((3, D), seed + 10, 0, 0.02)
        for i, (n, m) in enumerate((("bo", D), ("b1", FF), ("b2", D))):
            h[n] = randn_f16((m,), seed + 13 + i, 0, 0.02)
        for i, n in enumerate(("g1", "g2")):
            h[n] = randn_f16((D,), seed + 20 + i, 1.0, 0.02)
        for i, n in enumerate(("be1", "be2")):
            h[n] = randn_f16((D,), seed + 22 + i, 0.0, 0.02)
        d = self.d = {k: dev(v) for k, v in h.items()}
        for n in ("h1", "a", "o", "h2", "y"):
            d[n] = torch.empty((T, D), dtype=f16, device="cuda")
        d["qkv"] = torch.empty((3, T, D), dtype=f16, device="cuda")
        d["f"] = torch.empty((T, FF), dtype=f16, device="cuda")
        p = lambda n: d[n].data_ptr()

        # per-op scratch, as the reference's bump workspace hands it out (split-K planes of the narrow linears)
        ws_bytes = max(lib.mi_gemm_f16_workspace(T, K_, F_, L.W_KF, 1) for (K_, F_) in ((D, D), (D, FF), (FF, D)))
        self.ws = torch.empty(max(ws_bytes, 256), dtype=torch.uint8, device="cuda")
        wsp = self.ws.data_ptr()

        # The two norms are folded into the linears that read them, once, as a model would at load
        # (mi_lnfold_prepare_f16): gamma into the weights' rows, beta into the bias, column sums for the mean's term.
        f32 = torch.float32
        d["wqkv_p"], d["w1_p"] = torch.empty_like(d["wqkv"]), torch.empty_like(d["w1"])
        d["cs_qkv"], d["bp_qkv"] = (torch.empty((3, D), dtype=f32, device="cuda") for _ in range(2))
        d["cs_1"], d["bp_1"] = (torch.empty((FF,), dtype=f32, device="cuda") for _ in range(2))
        nseg = (D + 31) // 32
        d["st_x"], d["st_o"] = (torch.empty((nseg, T, 2), dtype=f32, device="cuda") for _ in range(2))
        for i in range(3):
            rc = lib.mi_lnfold_prepare_f16(d["wqkv_p"][i].data_ptr(), d["cs_qkv"][i].data_ptr(), d["bp_qkv"][i].data_ptr(), d["wqkv"][i].data_ptr(),
                                           p("g1"), p("be1"), d["bqkv"][i].data_ptr(), D, D, D, L.W_KF, stream)
            assert rc == 0, rc
        rc = lib.mi_lnfold_prepare_f16(p("w1_p"), p("cs_1"), p("bp_1"), p("w1"), p("g2"), p("be2"), p("b1"), D, FF, FF, L.W_KF, stream)
        assert rc == 0, rc
        torch.cuda.synchronize()
        self._lib, self._wsp, self._ws_bytes = lib, wsp, ws_bytes
        self.calls_before_fc1, self.fc1, self.calls_after_fc1 = self.calls_on(stream)

    def calls_on(self, stream):
        """The block's seven launches bound to `stream`: (those before fc1, fc1, those after it)."""
        import numpy as np
        lib, L, wsp, ws_bytes = self._lib, self.L, self._wsp, self._ws_bytes
        T, D, H, E, FF = self.T, self.D, self.H, self.E, self.FF
        p = lambda n: self.d[n].data_ptr()

        def gemm(y, x, w, b, K, F, epi, res=None):
            return Call(lib.mi_gemm_f16, p(y), p(x), p(w), p(b), (p(res) if res else None), T, K, F, F, K, F,
                        L.W_KF, L.BIAS_COL, L.EPI[epi], L.F16, wsp, ws_bytes, stream)

        tok = L.strides4(1, D, E, T * D)      # (E, L, H, B) strides of a token-major [T][H][E] buffer
        scale = 1.0 / np.sqrt(E)
        before = [
            # row statistics of the block's input (inside a stack the previous block's last GEMM leaves them)
            Call(lib.mi_rowstats_f16, p("st_x"), p("x"), D, D, T, stream),
            # LN1 + the three projections, one batched launch on the raw rows (plane strides: Y T*D, W D*D, vectors D)
            Call(lib.mi_lnfold_gemm_f16, p("qkv"), None, p("x"), p("st_x"), 1e-5, p("wqkv_p"), p("cs_qkv"), p("bp_qkv"), None, 0.0,
                 T, D, D, D, D, D, L.W_KF, L.EPI["none"], L.F16, 3, T * D, D * D, D, None, 0, stream),
            Call(lib.mi_sdpa_f16, p("a"), L.F16, tok, p("qkv"), tok, p("qkv") + 2 * T * D, tok, p("qkv") + 4 * T * D, tok,
                 None, 0, None, None, E, T, T, H, 1, scale, None, 0, stream),
            # output projection + residual, leaving the row statistics of its result for LN2
            Call(lib.mi_gemm_rowstats_f16, p("o"), p("st_o"), p("a"), p("wo"), p("bo"), p("x"), 0.0, T, D, D, D, D,
                 L.W_KF, L.BIAS_COL, L.EPI["none"], wsp, ws_bytes, stream),
        ]
        # LN2 + fc1 + GELU on the raw rows of o
        fc1 = Call(lib.mi_lnfold_gemm_f16, p("f"), None, p("o"), p("st_o"), 1e-5, p("w1_p"), p("cs_1"), p("bp_1"), None, 0.0,
                   T, D, FF, FF, D, FF, L.W_KF, L.EPI["gelu"], L.F16, 1, 0, 0, 0, wsp, ws_bytes, stream)
        return before, fc1, [gemm("y", "f", "w2", "b2", FF, D, "none", res="o")]

    def check_against_unfolded(self):
        """The timed step's result against the same block with both norms run as ops of their own (mi_layernorm_f16, then
        the plain GEMMs): the parity gate of the tests, max relative error <= 1e-2 and cosine >= 0.9999."""
        import numpy as np
        import torch
        lib, L, wsp, ws_bytes = self._lib, self.L, self._wsp, self._ws_bytes
        T, D, H, E, FF = self.T, self.D, self.H, self.E, self.FF
        d = self.d
        p = lambda n: d[n].data_ptr()
        d["y_ref"] = torch.empty_like(d["y"])
        st = torch.cuda.current_stream().cuda_stream
        tok = L.strides4(1, D, E, T * D)

        def gemm(y, x, w, b, K, F, epi, res=None):
            return Call(lib.mi_gemm_f16, p(y), p(x), p(w), p(b), (p(res) if res else None), T, K, F, F, K, F,
                        L.W_KF, L.BIAS_COL, L.EPI[epi], L.F16, wsp, ws_bytes, st)
        for c in [Call(lib.mi_layernorm_f16, p("h1"), None, None, p("x"), p("g1"), p("be1"), D, T, 1e-5, st),
                  Call(lib.mi_gemm_f16_batched, p("qkv"), p("h1"), p("wqkv"), p("bqkv"), None, T, D, D, D, D, D,
                       L.W_KF, L.BIAS_COL, L.EPI["none"], L.F16, 3, T * D, 0, D * D, D, None, 0, st),
                  Call(lib.mi_sdpa_f16, p("a"), L.F16, tok, p("qkv"), tok, p("qkv") + 2 * T * D, tok, p("qkv") + 4 * T * D, tok,
                       None, 0, None, None, E, T, T, H, 1, 1.0 / np.sqrt(E), None, 0, st),
                  gemm("o", "a", "wo", "bo", D, D, "none", res="x"),
                  Call(lib.mi_layernorm_f16, p("h2"), None, None, p("o"), p("g2"), p("be2"), D, T, 1e-5, st),
                  gemm("f", "h2", "w1", "b1", D, FF, "gelu"),
                  gemm("y_ref", "f", "w2", "b2", FF, D, "none", res="o")]:
            c()
        self.step()
        torch.cuda.synchronize()
        # the update the block adds to the residual stream, not the stream itself (which alone would pass a loose gate)
        got = (d["y"].float() - d["x"].float()).double().flatten()
        want = (d["y_ref"].float() - d["x"].float()).double().flatten()
        max_rel = float((got - want).abs().max() / want.abs().max())
        cos = float(torch.dot(got, want) / (got.norm() * want.norm()))
        if not (max_rel <= 1e-2 and cos >= 0.9999):
            raise RuntimeError(f"folded block differs from the unfolded one: max_rel {max_rel:.3e}, cosine {cos:.6f}")
        return {"max_rel_vs_unfolded_block": round(max_rel, 6), "cosine_vs_unfolded_block": round(cos, 7)}

    def captured(self):
        """The block step captured as one HIP graph (its launches issued on the capturing stream)."""
        import torch
        g = torch.cuda.CUDAGraph()
        with torch.cuda.graph(g):
            before, fc1, after = self.calls_on(torch.cuda.current_stream().cuda_stream)
            for c in before + [fc1] + after:
                c()
        return g

    def step(self, ev=None, ev_fc2=None):
        for c in self.calls_before_fc1:
            c()
        if ev is not None:
            ev[0].record()
        self.fc1()
        if ev is not None:
            ev[1].record()
            ev[2].record()       # nothing between ev[1] and ev[2]: what one event marker itself costs on this stream
        if ev_fc2 is not None:
            ev_fc2[0].record()
        for c in self.calls_after_fc1:      # the one launch after fc1 is fc2
            c()
        if ev_fc2 is not None:
            ev_fc2[1].record()
            ev_fc2[2].record()

    # ---- the same block on the CPU oracle, on a sample of the work, scaled to one block
    def cpu_baseline(self):
        import numpy as np
        import oracle
        h = self.host
        T, D, H, E = self.T, self.D, self.H, self.E
        # One whole block: every token row through the six linears and both layer norms, all 20 heads of
        # the three-pass attention at full length (a few seconds on 16 threads), repeated `reps` times.
        reps = 3
        rows, heads = T, H
        qa, ka, va = (randn_f16((1, heads, T, E), sd) for sd in (5, 6, 7))
        t_lin = t_att = 0.0
        for _ in range(reps):
            t0 = time.perf_counter()
            x = h["x"][:rows]
            h1, _, _ = oracle.layernorm_f16(x, h["g1"], h["be1"], 1e-5)
            q = oracle.gemm_f16(h1, h["wqkv"][0], h["bqkv"][0])
            oracle.gemm_f16(h1, h["wqkv"][1], h["bqkv"][1])
            oracle.gemm_f16(h1, h["wqkv"][2], h["bqkv"][2])
            o = oracle.gemm_f16(q, h["wo"], h["bo"], residual=x)
            h2, _, _ = oracle.layernorm_f16(o, h["g2"], h["be2"], 1e-5)
            f = oracle.gemm_f16(h2, h["w1"], h["b1"], epi="gelu")
            oracle.gemm_f16(f, h["w2"], h["b2"], residual=o)
            t1 = time.perf_counter()
            oracle.sdpa_threepass_f16(qa, ka, va)
            t2 = time.perf_counter()
            t_lin += (t1 - t0) / reps
            t_att += (t2 - t1) / reps
        sec = t_lin + t_att
        return {
            "value": round(self.FLOP / sec / 1e12, 6), "unit": "TFLOP/s", "cores": oracle.threads(), "kind": "port",
            "sample": f"the whole block, {reps} times: all {T} token rows through the six linears + both layer norms "
                      f"({t_lin:.2f} s) and all {H} heads of the three-pass attention ({t_att:.2f} s) per block",
            "ms_per_step": round(sec * 1e3, 1),
        }


# ----------------------------------------------------------------------------- other configs (detail)

def decoder_layer_case(bsz, layout="kf", steps=200):
    """One Whisper-decoder-shaped layer per token (d 1280, 20x64 heads, FFN 5120, self cache 448 with the
    position at its end, cross cache 1500), weights in the reference's hoisted [K][F] layout: the eager step
    (Python host + one launch per kernel) and the same step replayed as a captured graph."""
    import time
    import torch
    import juliavision_amd as jv
    from juliavision_amd.decode import DecodeBuffers, DecoderLayerWeights, KVCache, StepGraph, decoder_layer_step
    d, H, E, ffn = 1280, 20, 64, 5120
    ctx = jv.Ctx("cuda")
    f16 = torch.float16
    w = (lambda k, f: torch.randn((k, f), dtype=f16, device="cuda") * 0.02) if layout == "kf" else \
        (lambda k, f: (torch.randn((f, k), dtype=f16, device="cuda") * 0.02).t())
    v = lambda n, m=0.0: torch.randn((n,), dtype=f16, device="cuda") * 0.02 + m
    W = DecoderLayerWeights(v(d, 1.0), v(d), w(d, 3 * d), v(3 * d), w(d, d), v(d), v(d, 1.0), v(d), w(d, d), v(d), w(d, d), v(d),
                            v(d, 1.0), v(d), w(d, ffn), v(ffn), w(ffn, d), v(d))
    cache = KVCache(1, bsz, H, E)
    for t in (cache.self_k, cache.self_v, cache.cross_k, cache.cross_v):
        t.normal_()
    buf = DecodeBuffers(bsz, d, ffn)
    x = torch.randn((bsz, d), dtype=f16, device="cuda")
    y = torch.empty_like(x)

    def step():                                  # the position advances once per token, not per layer: decode_step_case has it
        decoder_layer_step(ctx, W, cache, 0, x, y, buf)

    def timed(fn):
        cache.length.fill_(448)                  # every step writes slot 447 and attends the full 448-slot cache
        for _ in range(10):
            fn()
        torch.cuda.synchronize()
        t0 = time.perf_counter()
        for _ in range(steps):
            fn()
        torch.cuda.synchronize()
        return (time.perf_counter() - t0) / steps

    eager = timed(step)
    graph = StepGraph(step)
    replay = timed(graph.replay)
    weights = 2.0 * (3 * d * d + 3 * d * d + 2 * d * ffn)
    kv = 2.0 * 2 * bsz * H * E * (448 + 1500)
    return {"eager_us": round(eager * 1e6, 1), "graph_us": round(replay * 1e6, 1), "launches": (14 if layout == "kf" else 8) + (3 if bsz > (8 if layout == "fk" else 4) else 0),
            "GB/s_graph": round((weights + kv) / replay / 1e9, 1), "frac_hbm_peak_graph": round((weights + kv) / replay / 1e9 / PEAK_HBM_GBS, 4)}


def decode_step_case(steps=100):
    """A whole Whisper-large-v3-turbo-shaped decoder token at batch 1: 4 layers (as decoder_layer_case, [F][K]
    weights), final layer norm folded into the 1280 -> 51866 vocabulary projection, one graph replay per token.
    The reference's figure for the same step is 13.5 ms per token in fp32 on its card, against a 2.07 ms floor
    set by 634 MB of fp32 weights (WhisperRunner/src/decode.jl:18-24); here a token reads 290 MB of fp16."""
    import time
    import torch
    import juliavision_amd as jv
    from juliavision_amd.decode import DecodeBuffers, DecoderLayerWeights, KVCache, StepGraph, decoder_layer_step
    d, H, E, ffn, NL, V = 1280, 20, 64, 5120, 4, 51866
    ctx = jv.Ctx("cuda")
    f16 = torch.float16
    w = lambda k, f: (torch.randn((f, k), dtype=f16, device="cuda") * 0.02).t()
    v = lambda n, m=0.0: torch.randn((n,), dtype=f16, device="cuda") * 0.02 + m
    layers = [DecoderLayerWeights(v(d, 1.0), v(d), w(d, 3 * d), v(3 * d), w(d, d), v(d), v(d, 1.0), v(d), w(d, d), v(d), w(d, d), v(d),
                                  v(d, 1.0), v(d), w(d, ffn), v(ffn), w(ffn, d), v(d)) for _ in range(NL)]
    lnf_g, lnf_b, wv = v(d, 1.0), v(d), w(d, V)
    cache = KVCache(NL, 1, H, E)
    for t in (cache.self_k, cache.self_v, cache.cross_k, cache.cross_v):
        t.normal_()
    buf = DecodeBuffers(1, d, ffn)
    xs = [torch.randn((1, d), dtype=f16, device="cuda") for _ in range(NL + 1)]
    logits = torch.empty((1, V), dtype=torch.float32, device="cuda")

    def step():
        cache.advance(ctx)
        for i in range(NL):
            decoder_layer_step(ctx, layers[i], cache, i, xs[i], xs[i + 1], buf)
        ctx.ws.reset()
        jv.ln_matmul_(ctx, logits, wv, xs[NL], lnf_g, lnf_b, 1e-5)

    def timed(fn):
        cache.length.fill_(447)
        for _ in range(5):
            fn()
        torch.cuda.synchronize()
        t0 = time.perf_counter()
        for _ in range(steps):
            fn()
        torch.cuda.synchronize()
        return (time.perf_counter() - t0) / steps

    eager = timed(step)
    graph = StepGraph(step)
    replay = timed(graph.replay)
    if not bool(torch.isfinite(logits).all()):
        raise RuntimeError("decode step produced non-finite logits")
    nbytes = NL * 2.0 * (3 * d * d + 3 * d * d + 2 * d * ffn) + 2.0 * d * V + NL * 2.0 * 2 * H * E * (448 + 1500)
    return {"eager_us": round(eager * 1e6, 1), "graph_us": round(replay * 1e6, 1), "launches": 1 + NL * 8 + 1,
            "MB_per_token": round(nbytes / 1e6, 1), "GB/s_graph": round(nbytes / replay / 1e9, 1),
            "frac_hbm_peak_graph": round(nbytes / replay / 1e9 / PEAK_HBM_GBS, 4)}


def vit_encoder_case(steps=50):
    """BASELINE config 3 as a whole: ViT-S/14 at 518 x 518 (patch embedding as convolution-as-GEMM, class token and
    position embedding, 12 pre-LN blocks of 1370 tokens x 384 with 6 x 64 heads and a 1536 MLP, final norm), eager
    and replayed as one captured graph.  92.78 GFLOP in the blocks + 0.62 in the patch embedding."""
    import time
    import torch
    import juliavision_amd as jv
    from juliavision_amd.decode import StepGraph
    from juliavision_amd.encoder import EncoderLayerWeights, ViTEncoder, ViTWeights
    d, H, ffn, P, S, NL = 384, 6, 1536, 14, 518, 12
    T = 1 + 37 * 37
    ctx = jv.Ctx("cuda")
    f16 = torch.float16
    w = lambda k, f: torch.randn((k, f), dtype=f16, device="cuda") * 0.02
    v = lambda n, m=0.0: torch.randn((n,), dtype=f16, device="cuda") * 0.02 + m
    layers = [EncoderLayerWeights(v(d, 1.0), v(d), w(d, 3 * d), v(3 * d), w(d, d), v(d), v(d, 1.0), v(d), w(d, ffn), v(ffn), w(ffn, d), v(d))
              for _ in range(NL)]
    W = ViTWeights(torch.randn((d, 3, P, P), dtype=f16, device="cuda") * 0.02, v(d), w(1, d), w(T, d), layers, v(d, 1.0), v(d))
    enc = ViTEncoder(W, (S, S), H, ffn, fold_norms=ctx)      # the block norms folded into the linears that read them: 5 launches a block
    image = torch.rand((1, 3, S, S), dtype=f16, device="cuda")

    def timed(fn):
        for _ in range(5):
            fn()
        torch.cuda.synchronize()
        t0 = time.perf_counter()
        for _ in range(steps):
            fn()
        torch.cuda.synchronize()
        return (time.perf_counter() - t0) / steps

    run = lambda: enc(ctx, image)
    eager = timed(run)
    embed = timed(lambda: enc.embed(ctx, image))
    graph = StepGraph(run)
    replay = timed(graph.replay)
    if not bool(torch.isfinite(enc.out).all()):
        raise RuntimeError("ViT encoder produced non-finite output")
    flop = NL * (2.0 * T * d * (3 * d + d + 2 * ffn) + 4.0 * T * T * 64 * H) + 2.0 * (T - 1) * 588 * d
    return {"eager_ms": round(eager * 1e3, 4), "graph_ms": round(replay * 1e3, 4), "patch_embed_eager_us": round(embed * 1e6, 1),
            # 3 for the patch embedding, the row statistics of the tokens, five launches per block, the final norm
            "launches": 3 + 1 + 5 * NL + 1, "GFLOP": round(flop / 1e9, 2), "TFLOP/s_graph": round(flop / replay / 1e12, 1),
            "frac_mfma_peak_graph": round(flop / replay / 1e12 / PEAK_F16_TFLOPS, 4)}


def vit_graph_case(steps=50):
    """Config 3's encoder from its exported graph: a ViT-S/14 written the way DINOv2 -- the backbone of the reference's
    Depth Anything model -- is (class token concatenated in front, written-out attention, LayerScale), exported with
    torch.export on the host, converted to the reference's JSON schema, rewritten (graph.optimize) and run by the graph
    executor, eager and replayed as one captured graph.  Random weights; the same 93.39 GFLOP."""
    import time
    import torch
    import torch.nn as nn
    import juliavision_amd as jv
    from juliavision_amd import graph as G
    from juliavision_amd.decode import StepGraph
    d, H, P, S, NL = 384, 6, 14, 518, 12

    class Block(nn.Module):
        def __init__(self):
            super().__init__()
            self.norm1, self.norm2 = nn.LayerNorm(d, eps=1e-6), nn.LayerNorm(d, eps=1e-6)
            self.qkv, self.proj, self.fc1, self.fc2 = nn.Linear(d, 3 * d), nn.Linear(d, d), nn.Linear(d, 4 * d), nn.Linear(4 * d, d)
            self.ls1, self.ls2 = nn.Parameter(torch.ones(d)), nn.Parameter(torch.ones(d))

        def forward(self, x):
            B, N, C = x.shape
            qkv = self.qkv(self.norm1(x)).reshape(B, N, 3, H, C // H).permute(2, 0, 3, 1, 4)
            a = ((qkv[0] * (C // H) ** -0.5) @ qkv[1].transpose(-2, -1)).softmax(dim=-1)
            x = x + self.proj((a @ qkv[2]).transpose(1, 2).reshape(B, N, C)) * self.ls1
            return x + self.fc2(nn.functional.gelu(self.fc1(self.norm2(x)))) * self.ls2

    class ViT(nn.Module):
        def __init__(self):
            super().__init__()
            self.patch_embed = nn.Conv2d(3, d, P, P)
            self.cls_token, self.pos_embed = nn.Parameter(torch.zeros(1, 1, d)), nn.Parameter(torch.randn(1, 1 + (S // P) ** 2, d) * 0.02)
            self.blocks = nn.ModuleList([Block() for _ in range(NL)])
            self.norm = nn.LayerNorm(d, eps=1e-6)

        def forward(self, img):
            x = self.patch_embed(img).flatten(2).transpose(1, 2)
            x = torch.cat((self.cls_token.expand(x.shape[0], -1, -1), x), dim=1) + self.pos_embed
            for b in self.blocks:
                x = b(x)
            return self.norm(x)

    torch.manual_seed(0)
    m = ViT().eval().half()
    t0 = time.perf_counter()
    ep = torch.export.export(m, (torch.rand(1, 3, S, S).half(),)).run_decompositions()
    spec = G.convert(ep, "vit_s14")
    g = G.optimize(G.Graph.load(spec))
    host_s = time.perf_counter() - t0
    ctx = jv.Ctx("cuda")
    run = G.Executor(g, m.state_dict(), ctx)
    image = torch.rand((1, 3, S, S), dtype=torch.float16, device="cuda")

    def timed(fn):
        for _ in range(5):
            fn()
        torch.cuda.synchronize()
        t = time.perf_counter()
        for _ in range(steps):
            fn()
        torch.cuda.synchronize()
        return (time.perf_counter() - t) / steps

    step = lambda: run(image)
    eager = timed(step)
    replay = timed(StepGraph(step).replay)
    if not bool(torch.isfinite(run(image)).all()):
        raise RuntimeError("exported ViT produced non-finite output")
    try:                                              # context: the same module evaluated by torch itself
        tm = m.cuda()
        with torch.no_grad():
            torch_ms = round(timed(lambda: tm(image)) * 1e3, 4)
            agree = round(float((tm(image).float() - run(image).float()).abs().max() / tm(image).float().abs().max()), 5)
    except Exception as e:
        torch_ms, agree = type(e).__name__, None
    T = 1 + (S // P) ** 2
    flop = NL * (2.0 * T * d * (3 * d + d + 8 * d) + 4.0 * T * T * 64 * H) + 2.0 * (T - 1) * 588 * d
    return {"ops_exported": len(spec["ops"]), "ops_after_rewrites": len(g.ops), "export_and_rewrite_host_s": round(host_s, 2),
            "eager_ms": round(eager * 1e3, 4), "graph_ms": round(replay * 1e3, 4), "TFLOP/s_graph": round(flop / replay / 1e12, 1),
            "torch_eager_same_module_ms": torch_ms, "max_rel_diff_vs_torch": agree}


def whisper_graph_case(nl=32, steps=10):
    """Configs 1/2's model as a whole, from its exported graph: an audio encoder written the way Whisper large-v3's is
    (128 mel bins x 3000 frames through two 1-D convolutions with GELU, 1500 positions, `nl` pre-LN layers of
    d_model 1280 with 20 x 64 heads -- q_proj scaled by 1/8 ahead of a fused attention, k_proj without bias -- FFN 5120,
    the fp16 clamp after every layer, a final norm), exported on the meta device, converted, rewritten and run by the
    graph executor with random weights.  Reported per layer: what BASELINE's "ms per encoder block" is inside the model."""
    import time
    import torch
    import torch.nn as nn
    import torch.nn.functional as F
    import juliavision_amd as jv
    from juliavision_amd import graph as G
    from juliavision_amd.decode import StepGraph
    d, heads, mels, frames, ffn = 1280, 20, 128, 3000, 5120

    class Layer(nn.Module):
        def __init__(self):
            super().__init__()
            self.ln1, self.ln2 = nn.LayerNorm(d), nn.LayerNorm(d)
            self.q, self.k, self.v, self.o = nn.Linear(d, d), nn.Linear(d, d, bias=False), nn.Linear(d, d), nn.Linear(d, d)
            self.fc1, self.fc2 = nn.Linear(d, ffn), nn.Linear(ffn, d)

        def forward(self, x):
            B, T, D = x.shape
            y = self.ln1(x)
            sp = lambda t: t.view(B, T, heads, D // heads).transpose(1, 2)
            a = F.scaled_dot_product_attention(sp(self.q(y) * (D // heads) ** -0.5), sp(self.k(y)), sp(self.v(y)), scale=1.0)
            x = x + self.o(a.transpose(1, 2).reshape(B, T, D))
            x = x + self.fc2(F.gelu(self.fc1(self.ln2(x))))
            return torch.clamp(x, min=-64504.0, max=64504.0)

    class Encoder(nn.Module):
        def __init__(self):
            super().__init__()
            self.conv1, self.conv2 = nn.Conv1d(mels, d, 3, padding=1), nn.Conv1d(d, d, 3, stride=2, padding=1)
            self.pos = nn.Parameter(torch.empty(frames // 2, d))
            self.layers = nn.ModuleList([Layer() for _ in range(nl)])
            self.ln_post = nn.LayerNorm(d)

        def forward(self, mel):
            x = F.gelu(self.conv2(F.gelu(self.conv1(mel))))
            x = x.permute(0, 2, 1) + self.pos
            for layer in self.layers:
                x = layer(x)
            return self.ln_post(x)

    t0 = time.perf_counter()
    with torch.device("meta"):
        m = Encoder().eval().half()
        mel_meta = torch.empty(1, mels, frames, dtype=torch.float16)
    table = torch.export.default_decompositions()
    table.pop(torch.ops.aten.scaled_dot_product_attention.default, None)     # an accelerator export keeps the fused op
    spec = G.convert(torch.export.export(m, (mel_meta,)).run_decompositions(table), "whisper_encoder")
    g = G.optimize(G.Graph.load(spec))
    host_s = time.perf_counter() - t0
    torch.manual_seed(0)
    weights = {}
    for k, v in m.state_dict().items():
        norm_scale = k.endswith("weight") and v.dim() == 1
        weights[k] = torch.ones(v.shape, dtype=torch.float16, device="cuda") if norm_scale else \
            torch.randn(v.shape, dtype=torch.float16, device="cuda") * 0.02
    ctx = jv.Ctx("cuda")
    run = G.Executor(g, weights, ctx)
    mel = torch.randn((1, mels, frames), dtype=torch.float16, device="cuda")

    def timed(fn):
        for _ in range(3):
            fn()
        torch.cuda.synchronize()
        t = time.perf_counter()
        for _ in range(steps):
            fn()
        torch.cuda.synchronize()
        return (time.perf_counter() - t) / steps

    step = lambda: run(mel)
    eager = timed(step)
    replay = timed(StepGraph(step).replay)
    if not bool(torch.isfinite(run(mel)).all()):
        raise RuntimeError("exported Whisper-like encoder produced non-finite output")
    # context: the same module with the same weights evaluated by torch itself (vendor kernels, eager dispatch)
    try:
        tm = m.to_empty(device="cuda")
        tm.load_state_dict(weights)
        with torch.no_grad():
            torch_ms = round(timed(lambda: tm(mel)) * 1e3, 3)
            agree = float((tm(mel).float() - run(mel).float()).abs().max() / tm(mel).float().abs().max())
        del tm
    except Exception as e:
        torch_ms, agree = type(e).__name__, None
    T = frames // 2
    flop = nl * (2.0 * T * d * (4 * d + 2 * ffn) + 4.0 * T * T * 64 * heads) + 2.0 * frames * (3 * mels) * d + 2.0 * T * (3 * d) * d
    return {"layers": nl, "ops_exported": len(spec["ops"]), "ops_after_rewrites": len(g.ops), "export_and_rewrite_host_s": round(host_s, 2),
            "eager_ms": round(eager * 1e3, 3), "graph_ms": round(replay * 1e3, 3), "graph_ms_per_layer": round(replay * 1e3 / nl, 4),
            "torch_eager_same_module_ms": torch_ms, "max_rel_diff_vs_torch": None if agree is None else round(agree, 5),
            "GFLOP": round(flop / 1e9, 1), "TFLOP/s_graph": round(flop / replay / 1e12, 1),
            "frac_mfma_peak_graph": round(flop / replay / 1e12 / PEAK_F16_TFLOPS, 4)}


def decoder_graph_case(steps=100):
    """Config 5's model as a whole, from its exported graph: a decoder step written the way the reference's export wrapper
    writes Whisper-large-v3-turbo's (tools/export_whisper_decoder.py:90-240: token + position embedding, the
    arange <= cache_position mask, 4 pre-LN layers of d_model 1280 with 20 x 64 heads whose new K/V rows go into a
    448-slot cache by index_copy, cross-attention over 1500 precomputed states, FFN 5120, final norm, logits through the
    tied 51866 x 1280 embedding, caches returned through stack), exported on the meta device, converted, rewritten --
    the functional cache update becomes the in-place one, the mask a key count -- and replayed as one captured graph."""
    import time
    import torch
    import torch.nn as nn
    import torch.nn.functional as F
    import juliavision_amd as jv
    from juliavision_amd import graph as G
    from juliavision_amd.decode import StepGraph
    d, H, ffn, NL, V, T, S = 1280, 20, 5120, 4, 51866, 448, 1500
    hd = d // H

    class Layer(nn.Module):
        def __init__(self):
            super().__init__()
            self.ln1, self.ln2, self.ln3 = nn.LayerNorm(d), nn.LayerNorm(d), nn.LayerNorm(d)
            self.q, self.k, self.v, self.o = nn.Linear(d, d), nn.Linear(d, d, bias=False), nn.Linear(d, d), nn.Linear(d, d)
            self.cq, self.co = nn.Linear(d, d), nn.Linear(d, d)
            self.fc1, self.fc2 = nn.Linear(d, ffn), nn.Linear(ffn, d)

    class Step(nn.Module):
        def __init__(self):
            super().__init__()
            self.embed_tokens, self.embed_positions = nn.Embedding(V, d), nn.Embedding(T, d)
            self.layers = nn.ModuleList([Layer() for _ in range(NL)])
            self.layer_norm = nn.LayerNorm(d)

        def forward(self, ids, self_k, self_v, cross_k, cross_v, cache_position):
            B = self_k.shape[1]
            h = self.embed_tokens(ids) + self.embed_positions.weight[cache_position]
            idx = torch.arange(T, device=h.device)
            lowest = torch.full((), torch.finfo(h.dtype).min, dtype=h.dtype, device=h.device)
            mask = torch.where(idx <= cache_position, torch.zeros((), dtype=h.dtype, device=h.device), lowest).view(1, 1, 1, T).expand(B, H, 1, T)
            heads = lambda t: t.view(B, 1, H, hd).transpose(1, 2)
            newk, newv = [], []
            for i, l in enumerate(self.layers):
                r, h = h, l.ln1(h)
                q = heads(l.q(h) * hd ** -0.5)
                K_ = self_k[i].index_copy(2, cache_position, heads(l.k(h)))
                V_ = self_v[i].index_copy(2, cache_position, heads(l.v(h)))
                newk.append(K_)
                newv.append(V_)
                h = r + l.o(F.scaled_dot_product_attention(q, K_, V_, attn_mask=mask, scale=1.0).transpose(1, 2).reshape(B, 1, d))
                r, h = h, l.ln2(h)
                o = F.scaled_dot_product_attention(heads(l.cq(h) * hd ** -0.5), cross_k[i], cross_v[i], scale=1.0)
                h = r + l.co(o.transpose(1, 2).reshape(B, 1, d))
                r, h = h, l.ln3(h)
                h = r + l.fc2(F.gelu(l.fc1(h)))
            return F.linear(self.layer_norm(h), self.embed_tokens.weight), torch.stack(newk), torch.stack(newv)

    t0 = time.perf_counter()
    with torch.device("meta"):
        m = Step().eval().half()
        z = lambda *sh: torch.empty(*sh, dtype=torch.float16)
        args = (torch.empty(1, 1, dtype=torch.long), z(NL, 1, H, T, hd), z(NL, 1, H, T, hd), z(NL, 1, H, S, hd), z(NL, 1, H, S, hd),
                torch.empty(1, dtype=torch.long))
    table = torch.export.default_decompositions()
    table.pop(torch.ops.aten.scaled_dot_product_attention.default, None)     # an accelerator export keeps the fused op
    spec = G.convert(torch.export.export(m, args).run_decompositions(table), "whisper_decoder_step")
    g = G.optimize(G.Graph.load(spec))
    host_s = time.perf_counter() - t0
    if sum(o["aten"] == "sdpa_append" for o in g.ops) != NL:
        raise RuntimeError("the exported step's cache update did not fold: " + "; ".join(g.notes[-5:]))
    torch.manual_seed(0)
    weights = {}
    for k, v in m.state_dict().items():
        norm_scale = k.endswith("weight") and v.dim() == 1
        weights[k] = torch.ones(v.shape, dtype=torch.float16, device="cuda") if norm_scale else \
            torch.randn(v.shape, dtype=torch.float16, device="cuda") * 0.02
    ctx = jv.Ctx("cuda")
    run = G.Executor(g, weights, ctx)
    f16 = torch.float16
    ids = torch.randint(0, V, (1, 1), device="cuda")
    sk, sv = (torch.randn(NL, 1, H, T, hd, dtype=f16, device="cuda") for _ in range(2))
    ck, cv = (torch.randn(NL, 1, H, S, hd, dtype=f16, device="cuda") for _ in range(2))
    pos = torch.tensor([T - 1], device="cuda")                       # the last slot: every step attends the full cache

    def timed(fn):
        for _ in range(5):
            fn()
        torch.cuda.synchronize()
        t = time.perf_counter()
        for _ in range(steps):
            fn()
        torch.cuda.synchronize()
        return (time.perf_counter() - t) / steps

    step = lambda: run(ids, sk, sv, ck, cv, pos)
    eager = timed(step)
    replay = timed(StepGraph(step).replay)
    logits, nk, _ = run(ids, sk, sv, ck, cv, pos)
    if not bool(torch.isfinite(logits).all()) or nk.data_ptr() != sk.data_ptr():
        raise RuntimeError("exported decoder step: non-finite logits, or the returned cache is not the caller's")
    mb = 2.0 * (NL * (3 * d * d + 3 * d * d + 2 * d * ffn) + V * d) + 2.0 * 2 * H * hd * (T + S) * NL
    return {"layers": NL, "ops_exported": len(spec["ops"]), "launches_after_rewrites": len(g.ops), "export_and_rewrite_host_s": round(host_s, 2),
            "eager_us": round(eager * 1e6, 1), "graph_us": round(replay * 1e6, 1), "MB_per_token": round(mb / 1e6, 1),
            "GB/s_graph": round(mb / replay / 1e9, 1), "frac_hbm_peak_graph": round(mb / replay / 1e9 / PEAK_HBM_GBS, 4)}


def encoder_stack_case(nl=4, steps=50):
    """BASELINE config 2's block as it occurs in a stack: `nl` Whisper-shaped blocks in sequence (1500 x 1280, 20 x 64
    heads, FFN 5120, [K][F] weights), five launches each: the norms are folded into the linears that read them, the GEMMs
    that write the residual stream leave its row statistics behind.  Reported per block."""
    import time
    import torch
    import juliavision_amd as jv
    from juliavision_amd.decode import StepGraph
    from juliavision_amd.encoder import EncoderBuffers, EncoderLayerWeights, FoldedStats, encoder_layer_folded, fold_layer_norms
    T, d, H, ffn = 1500, 1280, 20, 5120
    ctx = jv.Ctx("cuda")
    f16 = torch.float16
    w = lambda k, f: torch.randn((k, f), dtype=f16, device="cuda") * 0.02
    v = lambda n, m=0.0: torch.randn((n,), dtype=f16, device="cuda") * 0.02 + m
    layers = [EncoderLayerWeights(v(d, 1.0), v(d), w(d, 3 * d), v(3 * d), w(d, d), v(d), v(d, 1.0), v(d), w(d, ffn), v(ffn), w(ffn, d), v(d))
              for _ in range(nl)]
    buf = EncoderBuffers(T, d, ffn)
    xs = [torch.randn((T, d), dtype=f16, device="cuda") for _ in range(2)]
    x0 = torch.randn((T, d), dtype=f16, device="cuda")

    folded = [fold_layer_norms(ctx, lw) for lw in layers]
    st = FoldedStats(T, d)

    def run():
        src = x0
        jv.rowstats_(ctx, st.x, x0)
        for i, fw in enumerate(folded):
            dst = xs[i % 2]
            encoder_layer_folded(ctx, fw, src, dst, buf, st, H, 1e-5, stats_out=i + 1 < nl)
            src = dst

    def timed(fn):
        for _ in range(5):
            fn()
        torch.cuda.synchronize()
        t0 = time.perf_counter()
        for _ in range(steps):
            fn()
        torch.cuda.synchronize()
        return (time.perf_counter() - t0) / steps

    eager = timed(run)
    replay = timed(StepGraph(run).replay)
    if not bool(torch.isfinite(xs[(nl - 1) % 2]).all()):
        raise RuntimeError("encoder stack produced non-finite output")
    flop = EncoderBlock.FLOP
    return {"blocks": nl, "eager_ms_per_block": round(eager / nl * 1e3, 4), "graph_ms_per_block": round(replay / nl * 1e3, 4),
            "launches": 1 + 5 * nl, "TFLOP/s_graph": round(flop * nl / replay / 1e12, 1),
            "frac_mfma_peak_graph": round(flop * nl / replay / 1e12 / PEAK_F16_TFLOPS, 4)}


def vendor_probe():
    """The same shapes through the libraries this image ships (hipBLASLt / rocBLAS behind torch.addmm and F.linear, the
    fused attention behind F.scaled_dot_product_attention, MIOpen behind F.conv2d), timed the same way with rotating
    buffers: context for the figures above, not part of the product path and not a baseline this build is scored on."""
    import torch
    import torch.nn.functional as F
    f16, out = torch.float16, {}
    r = lambda *sh: torch.randn(sh, dtype=f16, device="cuda")

    def timed(make, n=3, reps=20):
        fns = [make() for _ in range(n)]
        state = {"i": 0}

        def fn():
            fns[state["i"] % n]()
            state["i"] += 1
        med, lo, _ = event_time(fn, reps)
        return round(med * 1e6, 2), round(lo * 1e6, 2)

    def linear_kf():
        x, w, b = r(1500, 1280) / 36, r(1280, 5120) * 0.02, r(5120) * 0.02
        y = torch.empty((1500, 5120), dtype=f16, device="cuda")
        return lambda: torch.addmm(b, x, w, out=y)

    def linear_fk():
        x, w, b = r(1500, 1280) / 36, r(5120, 1280) * 0.02, r(5120) * 0.02
        return lambda: F.linear(x, w, b)

    def attn(B, H, Lq, E):
        def make():
            q, k, v = r(B, H, Lq, E), r(B, H, Lq, E), r(B, H, Lq, E)
            return lambda: F.scaled_dot_product_attention(q, k, v)
        return make

    def conv(channels_last):
        def make():
            x, w, b = r(1, 256, 64, 64), r(256, 256, 3, 3) * 0.02, r(256) * 0.02
            if channels_last:
                x, w = x.contiguous(memory_format=torch.channels_last), w.contiguous(memory_format=torch.channels_last)
            return lambda: F.conv2d(x, w, b, padding=1)
        return make

    for name, make in (("c1_linear_W[K][F]_torch_addmm", linear_kf), ("c1_linear_W[F][K]_torch_linear", linear_fk),
                       ("c2_attn_L1500_20x64_torch_sdpa", attn(1, 20, 1500, 64)), ("c4_attn_L4096_16x64_torch_sdpa", attn(1, 16, 4096, 64)),
                       ("sam2_global_attn_L4096_8x72_torch_sdpa", attn(1, 8, 4096, 72)),
                       ("c4_conv3x3_torch_conv2d_nchw", conv(False)), ("c4_conv3x3_torch_conv2d_channels_last", conv(True))):
        try:
            med, lo = timed(make)
            out[name] = {"us": med, "us_min": lo}
        except Exception as e:                      # a library that refuses a shape is a result too
            out[name] = {"error": type(e).__name__}
    return out


def detail_benchmarks(lib, L, stream, only=None):
    import numpy as np
    import torch
    out = {}
    f16 = torch.float16
    NB = 3   # rotating buffer sets

    def gemm_case(name, T, K, F, layout, epi="none", sets=NB, reps=20):
        if only is not None and only not in name:
            return None
        Xs = [torch.randn((T, K), dtype=f16, device="cuda") / K ** 0.5 for _ in range(sets)]
        Ws = [torch.randn((K, F) if layout == L.W_KF else (F, K), dtype=f16, device="cuda") * 0.02 for _ in range(sets)]
        b = torch.randn((F,), dtype=f16, device="cuda") * 0.02
        Ys = [torch.empty((T, F), dtype=f16, device="cuda") for _ in range(min(sets, 3))]
        need = lib.mi_gemm_f16_workspace(T, K, F, layout, 1)
        ws = torch.empty(max(need, 256), dtype=torch.uint8, device="cuda")
        calls = [Call(lib.mi_gemm_f16, Ys[i % len(Ys)].data_ptr(), Xs[i].data_ptr(), Ws[i].data_ptr(), b.data_ptr(), None, T, K, F, F, K,
                      (F if layout == L.W_KF else K), layout, L.BIAS_COL, L.EPI[epi], L.F16, ws.data_ptr(), need, stream) for i in range(sets)]
        state = {"i": 0}

        def fn():
            calls[state["i"] % sets]()
            state["i"] += 1
        med, lo, hi = event_time(fn, reps)
        flop = 2.0 * T * K * F
        wbytes = 2.0 * K * F
        out[name] = {"us": round(med * 1e6, 2), "us_min": round(lo * 1e6, 2), "TFLOP/s": round(flop / med / 1e12, 1),
                     "frac_mfma_peak": round(flop / med / 1e12 / PEAK_F16_TFLOPS, 4),
                     "weight_GB/s": round(wbytes / med / 1e9, 1)}
        return out[name]

    def attn_case(name, B, H, Lq, Lk, E, kv_len=None, sets=NB, reps=10, mask=None):
        """mask: None, "pad" ((B,1,1,Lk) fp16 0 / finfo.min padding mask) or "full" (dense fp16 (B,H,Lq,Lk))."""
        if only is not None and only not in name:
            return
        qs = [torch.randn((B, H, Lq, E), dtype=f16, device="cuda") for _ in range(sets)]
        ks = [torch.randn((B, H, Lk, E), dtype=f16, device="cuda") for _ in range(sets)]
        vs = [torch.randn((B, H, Lk, E), dtype=f16, device="cuda") for _ in range(sets)]
        o = torch.empty((B, H, Lq, E), dtype=f16, device="cuda")
        kl = None if kv_len is None else torch.full((B,), kv_len, dtype=torch.int32, device="cuda")
        need = lib.mi_sdpa_f16_workspace(E, Lq, Lk, H, B, 0)
        ws = torch.empty(max(need, 256), dtype=torch.uint8, device="cuda")
        dq, dk = L.strides4(1, E, E * Lq, E * Lq * H), L.strides4(1, E, E * Lk, E * Lk * H)
        mk, mst = None, None
        if mask == "pad":
            mk = torch.zeros((B, 1, 1, Lk), dtype=f16, device="cuda")
            mk[..., Lk - 100:] = torch.finfo(f16).min
            mst = L.strides4(1, 0, 0, Lk)
        elif mask == "full":
            mk = torch.randn((B, H, Lq, Lk), dtype=f16, device="cuda")
            mst = L.strides4(1, Lk, Lk * Lq, Lk * Lq * H)
        calls = [Call(lib.mi_sdpa_f16, o.data_ptr(), L.F16, None, qs[i].data_ptr(), dq, ks[i].data_ptr(), dk, vs[i].data_ptr(), dk,
                      (mk.data_ptr() if mk is not None else None), L.F16, mst, (kl.data_ptr() if kl is not None else None), E, Lq, Lk, H, B, 1.0 / np.sqrt(E),
                      ws.data_ptr(), need, stream) for i in range(sets)]
        state = {"i": 0}

        def fn():
            calls[state["i"] % sets]()
            state["i"] += 1
        med, lo, hi = event_time(fn, reps)
        keys = Lk if kv_len is None else kv_len
        flop = 4.0 * Lq * keys * E * H * B
        kvbytes = 2.0 * 2 * keys * E * H * B
        out[name] = {"us": round(med * 1e6, 2), "us_min": round(lo * 1e6, 2), "TFLOP/s": round(flop / med / 1e12, 2),
                     "frac_mfma_peak": round(flop / med / 1e12 / PEAK_F16_TFLOPS, 4), "kv_GB/s": round(kvbytes / med / 1e9, 1)}

    # config 1: the linear, both weight layouts
    gemm_case("c1_linear_1500x1280x5120_W[K][F]_bias", 1500, 1280, 5120, L.W_KF)
    gemm_case("c1_linear_1500x1280x5120_W[F][K]_bias", 1500, 1280, 5120, L.W_FK)
    # not a BASELINE config: the same kernel family where the grid fills the chip for many rounds (256 x 256 tiles)
    gemm_case("square_4096x4096x4096_W[K][F]_bias", 4096, 4096, 4096, L.W_KF, sets=2, reps=10)
    gemm_case("square_8192x8192x8192_W[K][F]_bias", 8192, 8192, 8192, L.W_KF, sets=1, reps=5)
    gemm_case("c2_proj_1500x1280x1280", 1500, 1280, 1280, L.W_KF)
    gemm_case("c2_fc2_1500x5120x1280", 1500, 5120, 1280, L.W_KF)
    # config 3: ViT-S/14 shapes
    gemm_case("c3_qkv_1370x384x1152", 1370, 384, 1152, L.W_KF)
    gemm_case("c3_fc1_1370x384x1536", 1370, 384, 1536, L.W_KF, epi="gelu")
    gemm_case("c3_fc2_1370x1536x384", 1370, 1536, 384, L.W_KF)
    attn_case("c3_attn_L1370_6x64", 1, 6, 1370, 1370, 64)
    # other grids of more 32-query tiles than CUs and at most one 64-query tile per CU (ViT-B/16 at 1024 tokens, a half-width
    # Whisper encoder): the 64-query form whose key quarters share K and V through LDS, like config 3's
    attn_case("vit_attn_L1024_16x64", 1, 16, 1024, 1024, 64)
    attn_case("attn_L1500_10x64", 1, 10, 1500, 1500, 64)
    attn_case("c2_attn_L1500_20x64", 1, 20, 1500, 1500, 64)
    # the same attention with an additive mask: it stays in the fused kernel (the reference's fused plan declines masks)
    attn_case("c2_attn_L1500_20x64_padding_mask", 1, 20, 1500, 1500, 64, mask="pad")
    attn_case("c2_attn_L1500_20x64_dense_fp16_mask", 1, 20, 1500, 1500, 64, mask="full")
    # the reference's own SAM 2.1 attention shapes, head size 72: global blocks and 16 windows of 256 (tools/attn_lab.jl:8-14)
    attn_case("sam2_global_attn_L4096_8x72", 1, 8, 4096, 4096, 72)
    attn_case("sam2_window_attn_L256_8x72_b16", 16, 8, 256, 256, 72)
    # the reference's flash-decoding case: SAM 2.1's mask decoder, 23 queries over the 4096 image tokens, 8 heads of 16
    # (test_flash.jl:189-190; 0.4279 -> 0.1204 ms split six ways on its card, plans/STATUS.md:70-75)
    attn_case("sam2_decoder_cross_attn_Lq23_Lk4096_8x16", 1, 8, 23, 4096, 16)
    def conv_case():
        x = torch.randn((1, 256, 64, 64), dtype=f16, device="cuda")
        w = torch.randn((256, 256, 3, 3), dtype=f16, device="cuda") * 0.02
        b = torch.randn((256,), dtype=f16, device="cuda") * 0.02
        o = torch.empty((1, 256, 64, 64), dtype=f16, device="cuda")
        need = lib.mi_conv2d_f16_workspace(64, 64, 256, 1, 3, 3, 256, 1, 1, 1, 1, 1, 1)
        ws = torch.empty(max(need, 256), dtype=torch.uint8, device="cuda")
        conv = Call(lib.mi_conv2d_f16, o.data_ptr(), x.data_ptr(), w.data_ptr(), b.data_ptr(), 64, 64, 256, 1, 3, 3, 256,
                    1, 1, 1, 1, 1, 1, 1, L.EPI["none"], ws.data_ptr(), need, stream)
        med, lo, hi = event_time(conv, 10)
        flop = 2.0 * 4096 * 2304 * 256
        out["c4_conv3x3_256to256_64x64"] = {"us": round(med * 1e6, 2), "TFLOP/s": round(flop / med / 1e12, 2),
                                            "frac_mfma_peak": round(flop / med / 1e12 / PEAK_F16_TFLOPS, 4)}

    def conv_nhwc_case():
        # the same convolution over a channels-last map: the GEMM gathers its A operand from x, nothing is staged
        x = torch.randn((1, 64, 64, 256), dtype=f16, device="cuda")
        w = torch.randn((256, 3, 3, 256), dtype=f16, device="cuda") * 0.02
        b = torch.randn((256,), dtype=f16, device="cuda")
        o = torch.empty((1, 64, 64, 256), dtype=f16, device="cuda")
        geo = (64, 64, 256, 1, 3, 3, 256, 1, 1, 1, 1, 1, 1)
        need = lib.mi_conv2d_nhwc_f16_workspace(*geo)
        ws = torch.empty(max(need, 256), dtype=torch.uint8, device="cuda")
        conv = Call(lib.mi_conv2d_nhwc_f16, o.data_ptr(), x.data_ptr(), w.data_ptr(), b.data_ptr(), *geo, L.EPI["none"],
                    ws.data_ptr(), need, stream)
        med, lo, hi = event_time(conv, 10)
        flop = 2.0 * 4096 * 2304 * 256
        out["c4_conv3x3_256to256_64x64_nhwc"] = {"us": round(med * 1e6, 2), "TFLOP/s": round(flop / med / 1e12, 2),
                                                  "range_us": [round(lo * 1e6, 2), round(hi * 1e6, 2)]}

    def convt_case(name, Cin, Hi, Cout):
        # SAM 2's mask-decoder upsamplers: kernel 2, stride 2 (test_convtranspose_gemm.jl:36)
        if only is not None and only not in name:
            return
        x = torch.randn((1, Cin, Hi, Hi), dtype=f16, device="cuda")
        w = torch.randn((Cin, Cout, 2, 2), dtype=f16, device="cuda") * 0.05
        b = torch.randn((Cout,), dtype=f16, device="cuda") * 0.02
        o = torch.empty((1, Cout, 2 * Hi, 2 * Hi), dtype=f16, device="cuda")
        geo = (Hi, Hi, Cin, 1, 2, 2, Cout, 2, 2, 0, 0, 1, 1, 0, 0, 1)
        need = lib.mi_convtranspose2d_f16_workspace(*geo)
        ws = torch.empty(max(need, 256), dtype=torch.uint8, device="cuda")
        call = Call(lib.mi_convtranspose2d_f16, o.data_ptr(), x.data_ptr(), w.data_ptr(), b.data_ptr(), *geo, ws.data_ptr(), need, stream)
        med, lo, hi = event_time(call, 10)
        flop = 2.0 * Hi * Hi * Cin * Cout * 4
        io = 2.0 * (Cin * Hi * Hi + Cout * 4 * Hi * Hi + Cin * Cout * 4)
        out[name] = {"us": round(med * 1e6, 2), "us_min": round(lo * 1e6, 2), "TFLOP/s": round(flop / med / 1e12, 2),
                     "io_GB/s": round(io / med / 1e9, 1)}

    def decode_cases():
        # config 5: decode-sized linears (HBM-bound on the weights; enough rotating weight sets to exceed the
        # 256 MB last-level cache) and single-query attention over the caches
        for bsz in (1, 4, 8):
            for (K, F) in ((1280, 1280), (1280, 5120)):
                sets = int(np.ceil(320e6 / (2.0 * K * F)))
                for lay, tag in ((L.W_KF, "W[K][F]"), (L.W_FK, "W[F][K]")):
                    name = f"c5_linear_b{bsz}_{K}to{F}_{tag}"
                    if only is not None and only not in name:
                        continue
                    r = gemm_case(name, bsz, K, F, lay, sets=sets, reps=sets)
                    r["frac_hbm_peak"] = round(r["weight_GB/s"] / PEAK_HBM_GBS, 4)
                    del r["TFLOP/s"], r["frac_mfma_peak"]
            for (nm, Lk, kvl) in (("self_pos447", 448, 448), ("self_pos3", 448, 4), ("cross", 1500, None)):
                name = f"c5_attn_b{bsz}_{nm}"
                if only is not None and only not in name:
                    continue
                sets = int(np.ceil(320e6 / (4.0 * Lk * 64 * 20 * bsz)))
                attn_case(name, bsz, 20, 1, Lk, 64, kv_len=kvl, sets=sets, reps=sets)
                r = out[name]
                r["frac_hbm_peak"] = round(r["kv_GB/s"] / PEAK_HBM_GBS, 4)
                del r["TFLOP/s"], r["frac_mfma_peak"]

    # config 5, whole decoder layer per token: the per-op dispatch the reference is bound by
    # (~63 us per op, plans/whisper-decoder.md:161-166) against one graph launch of the same work
    for bsz in (1, 4, 8):
        for lay, tag in (("kf", "W[K][F]"), ("fk", "W[F][K]")):
            name = f"c5_decoder_layer_b{bsz}_{tag}"
            if only is None or only in name:
                out[name] = decoder_layer_case(bsz, lay)

    name = "c2_encoder_stack_4blocks"
    if only is None or only in name:
        out[name] = encoder_stack_case()

    name = "c3_vit_s14_518_encoder_12layers"
    if only is None or only in name:
        out[name] = vit_encoder_case()

    name = "c2_whisper_encoder_32layers_from_exported_graph"
    if only is None or only in name:
        out[name] = whisper_graph_case()

    name = "c3_vit_s14_518_from_exported_graph"
    if only is None or only in name:
        out[name] = vit_graph_case()

    name = "vendor_probe_same_shapes_through_torch"
    if only is None or only in name:
        out[name] = vendor_probe()

    name = "c5_decode_step_4layers_vocab51866_b1"
    if only is None or only in name:
        out[name] = decode_step_case()

    name = "c5_decode_step_from_exported_graph_b1"
    if only is None or only in name:
        out[name] = decoder_graph_case()

    # config 4: global attention at 4096 and the 3x3 conv
    attn_case("c4_attn_L4096_16x64", 1, 16, 4096, 4096, 64)
    if only is None or only in "c4_conv3x3_256to256_64x64":
        conv_case()
    if only is None or only in "c4_conv3x3_256to256_64x64_nhwc":
        conv_nhwc_case()
    convt_case("sam2_upsample_convT2x2_256to64_64x64", 256, 64, 64)
    convt_case("sam2_upsample_convT2x2_64to32_128x128", 64, 128, 32)
    decode_cases()
    if only is not None:
        return {k: v for k, v in out.items() if only in k}
    return out


# ----------------------------------------------------------------------------- main

def main():
    args = parse_args()
    if args.gpus != 1:
        print(f"bench.py: this build runs on one GPU; --gpus {args.gpus} is not supported (no collective, "
              "sharding or rank code exists in this path).", file=sys.stderr)
        sys.exit(2)
    import torch
    import juliavision_amd as jv
    L = jv._lib
    lib = L.init()
    stream = torch.cuda.current_stream().cuda_stream
    if args.calibrate_copy:
        src = torch.empty(256 << 20, dtype=torch.uint8, device="cuda").random_(0, 255)
        dst = torch.empty_like(src)
        for _ in range(3):
            lib.mi_probe_copy(dst.data_ptr(), src.data_ptr(), src.numel(), stream)
        torch.cuda.synchronize()
        del src, dst
    if args.phase_stamps:
        print(json.dumps({"phase_stamps": phase_stamps(lib, L, stream)}, indent=1))
        return
    if args.only is not None:
        print(json.dumps({"only": args.only, "detail": detail_benchmarks(lib, L, stream, args.only)}))
        return
    blk = EncoderBlock(lib, stream)
    agreement = blk.check_against_unfolded()

    for _ in range(args.warmup):
        blk.step()
    torch.cuda.synchronize()
    # The step the driver times is what the reference's runtime runs: the block's launches captured once and replayed
    # (Lava.capture / replay, execute.jl:18-92), so that the figure is the kernels and not the host's launch gaps.
    graph = blk.captured()
    # Warm-up until the clock has settled: the shader clock ramps up over the first milliseconds of load and then gives
    # way to the power limit; chunks of replays are timed until three in a row agree to 1 % (at most ~2 s).
    warm_chunks, chunk_ms = 0, []
    while warm_chunks < 200:
        torch.cuda.synchronize()
        c0 = time.perf_counter()
        for _ in range(64):
            graph.replay()
        torch.cuda.synchronize()
        chunk_ms.append((time.perf_counter() - c0) * 1e3 / 64)
        warm_chunks += 1
        if len(chunk_ms) >= 3 and max(chunk_ms[-3:]) <= 1.01 * min(chunk_ms[-3:]):
            break
    torch.cuda.synchronize()
    t0 = time.perf_counter()
    for i in range(args.steps):
        graph.replay()
    torch.cuda.synchronize()
    t1 = time.perf_counter()
    sec = (t1 - t0) / args.steps
    y = blk.d["y"].float()
    if not bool(torch.isfinite(y).all()) or float(y.abs().max()) < 1e-3:
        raise RuntimeError("encoder block produced non-finite or empty output")
    # the same steps issued eagerly (one C-ABI call per launch from Python), for the record
    torch.cuda.synchronize()
    e0 = time.perf_counter()
    for i in range(args.steps):
        blk.step()
    torch.cuda.synchronize()
    eager_sec = (time.perf_counter() - e0) / args.steps

    # The two largest launches of the step -- fc1 (config 1's shape + GELU) and fc2 -- bracketed by HIP events on the
    # launch stream in NSAMP eager steps after the timed loop (an event marker costs about 5 us of queue time, so
    # none sits inside the timed region).  [ev0, ev1] holds the kernel plus one marker, [ev1, ev2] one marker and
    # nothing else: their difference is the kernel's own duration.  `roofline` describes whichever of the two takes
    # longer; the other is reported beside it.
    NSAMP = max(15, min(args.steps, 64))
    ev1 = [tuple(torch.cuda.Event(enable_timing=True) for _ in range(3)) for _ in range(NSAMP)]
    ev2 = [tuple(torch.cuda.Event(enable_timing=True) for _ in range(3)) for _ in range(NSAMP)]
    for i in range(NSAMP):
        blk.step(ev1[i], ev2[i])
    torch.cuda.synchronize()

    def kernel_us(evs):
        d = sorted((e0.elapsed_time(e1) - e1.elapsed_time(e2)) * 1e3 for e0, e1, e2 in evs)
        br = sum(e0.elapsed_time(e1) for e0, e1, _ in evs) / len(evs) * 1e3
        mk = sum(e1.elapsed_time(e2) for _, e1, e2 in evs) / len(evs) * 1e3
        return {"avg": sum(d) / len(d), "median": d[len(d) // 2], "min": d[0], "bracket": br, "marker": mk}
    fc1_t, fc2_t = kernel_us(ev1), kernel_us(ev2)

    # Shader clock during the fc1 launch: workgroup 0 of the kernel stores {shader clock, 100 MHz clock} at its start
    # and end (mi_set_clock_probe), in a few untimed steps of their own.
    clk = torch.zeros(4, dtype=torch.int64, device="cuda")
    lib.mi_set_clock_probe(clk.data_ptr())
    mhz = []
    for _ in range(8):
        for c in blk.calls_before_fc1:
            c()
        blk.fc1()
        torch.cuda.synchronize()
        c0, r0, c1, r1 = (int(v) for v in clk.tolist())
        if r1 > r0:
            mhz.append((c1 - c0) / (r1 - r0) * 100.0)
        for c in blk.calls_after_fc1:
            c()
    lib.mi_set_clock_probe(None)
    torch.cuda.synchronize()
    shader_mhz = sorted(mhz)[len(mhz) // 2] if mhz else None
    probe = peak_probe(lib, stream)

    dominant = ("fc1", fc1_t, "gemm_w4_kernel<128,256,1,4,KN> fc1: Y[1500x5120] = gelu(LN(X)[1500x1280].W[1280x5120] + b), the layer norm folded into the store") \
        if fc1_t["avg"] >= fc2_t["avg"] else \
        ("fc2", fc2_t, "gemm_w4_kernel<128,128,2,2,KN,SK> fc2: Y[1500x1280] = X[1500x5120].W[5120x1280] + b + residual, "
                       "K in two slices exchanged inside the launch")
    other = ("fc2", fc2_t) if dominant[0] == "fc1" else ("fc1", fc1_t)
    dom_t = dominant[1]
    fc_avg = dom_t["avg"] * 1e-6
    achieved = blk.FC1_FLOP / fc_avg / 1e12          # fc1 and fc2 are the same 19.66 GFLOP
    cus = int(jv.caps().cores)
    peak_at_clock = cus * MFMA_FLOP_PER_CLK_PER_CU * shader_mhz * 1e6 / 1e12 if shader_mhz else None
    res = {
        "metric": "fp16 GEMM/attention TFLOP/s + % of MFMA peak; ms per encoder block",
        "value": round(blk.FLOP / sec / 1e12, 2),
        "unit": "TFLOP/s",
        "n_gpus": 1, "steps": args.steps, "warmup": args.warmup,
        "ms_per_step": round(sec * 1e3, 4),
        "higher_is_better": True, "scaling": "weak", "vs_baseline": None,
        "dtype": "f16", "data": "synthetic",
        "config": {"workload": "BASELINE config 2: Whisper-large-v3-turbo-shaped encoder block, batch 1, 1500 tokens, "
                               "d_model 1280, 20x64 heads, FFN 5120 GELU(erf), pre-LN, fp16 in / fp32 accumulate; "
                               "70.50 GFLOP per block (58.98 GEMM + 11.52 attention); 6 launches via the C ABI (row statistics "
                               "of the input, q/k/v behind the folded first norm, attention, projection + residual, GELU linear "
                               "behind the folded second norm, second MLP linear + residual), captured once and replayed as a HIP graph",
                   "tokens": 1500, "d_model": 1280, "heads": 20, "head_dim": 64, "ffn": 5120,
                   "weight_layout": "[K][F] (the reference's hoisted layout)"},
        "frac_mfma_peak": round(blk.FLOP / sec / 1e12 / PEAK_F16_TFLOPS, 4),
        "eager_ms_per_step": round(eager_sec * 1e3, 4),
        "agreement": agreement,
        "warmup_replays_until_clock_plateau": 64 * warm_chunks,
        "roofline": {"kernel": dominant[2], "launch": dominant[0],
                     "bound": "mfma", "achieved": round(achieved, 1), "peak": PEAK_F16_TFLOPS, "unit": "TFLOP/s",
                     "frac": round(achieved / PEAK_F16_TFLOPS, 4), "traffic": fc_traffic_bytes(dominant[0]),
                     "traffic_source": FC1_TRAFFIC_FILE,
                     # next to the vendor-peak fraction, never instead of it: what this box delivers with nothing in
                     # the way (measured in this run through mi_probe_mfma / mi_probe_copy), and the same rate against
                     # the MFMA units at the shader clock measured inside the fc1 launch
                     "mfma_only_tflops": probe["mfma_only_tflops"], "mfma_only_frac_of_peak": probe["mfma_only_frac_of_peak"],
                     "c1_no_memory_us": probe["c1_no_memory_us"], "launch_over_no_memory": round(dom_t["avg"] / probe["c1_no_memory_us"], 3),
                     "hbm_copy_gbs": probe["hbm_copy_gbs"],
                     "shader_clock_mhz": round(shader_mhz, 1) if shader_mhz else None,
                     "peak_at_measured_clock": round(peak_at_clock, 1) if peak_at_clock else None,
                     "frac_at_measured_clock": round(achieved / peak_at_clock, 4) if peak_at_clock else None,
                     "flop_per_launch": blk.FC1_FLOP, "avg_launch_us": round(dom_t["avg"], 2),
                     "median_launch_us": round(dom_t["median"], 2), "min_launch_us": round(dom_t["min"], 2),
                     "avg_event_bracket_us": round(dom_t["bracket"], 2),
                     "avg_event_marker_us": round(dom_t["marker"], 2),
                     "timed_launches": NSAMP,
                     "other_large_launch": {"launch": other[0], "avg_launch_us": round(other[1]["avg"], 2),
                                            "median_launch_us": round(other[1]["median"], 2),
                                            "frac": round(blk.FC1_FLOP / (other[1]["avg"] * 1e-6) / 1e12 / PEAK_F16_TFLOPS, 4)}},
        "peak_probe": probe,
    }
    if args.detail:
        res["detail"] = detail_benchmarks(lib, L, stream)
    if args.cpu:
        res["cpu_baseline"] = blk.cpu_baseline()
    else:
        res["cpu_baseline"] = None
    print(json.dumps(res))


if __name__ == "__main__":
    main()
