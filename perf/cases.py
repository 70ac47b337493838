"""The work whose speed is watched: what a program that uses this package has it do, through the public entry points.

Eight kinds of work.  ``linear``, ``attention``, ``conv`` and ``upsample`` are single calls as a host program issues them, one
after the other; ``encoder``, ``vit``, ``decode`` and ``exported`` are whole compositions, either issued call by call or
captured once and replayed (``replay``).  ``listed()`` names typical members, ``draw(rng)`` gives further ones of the
same ranges: sizes from the smallest calls to the largest, odd ones among them.

All data is fp16 with fp32 accumulation, the one data type of the path; fp32 results are drawn where the entry point has them.
"""
import functools
import math

import torch
import torch.nn as nn
import torch.nn.functional as F

import juliavision_amd as jv
from juliavision_amd import graph as G
from juliavision_amd.decode import DecodeBuffers, DecoderLayerWeights, KVCache, StepGraph, decoder_layer_step
from juliavision_amd.encoder import (EncoderBuffers, EncoderLayerWeights, FoldedStats, ViTEncoder, ViTWeights, encoder_layer_folded,
                                     fold_layer_norms)

F16 = torch.float16
PATCH = 14                      # the ViT cases: 14 x 14 patches, 384 features in 6 heads, an MLP of 1536
VIT_D, VIT_HEADS, VIT_FFN = 384, 6, 1536


# ----------------------------------------------------------------------------- the cases

def listed():
    return [
        # an MLP layer of a mask decoder: a couple of dozen tokens; what such a call costs is its launch
        {"name": "linear_small", "kind": "linear", "T": 23, "K": 256, "F": 2048, "layout": "fk", "epi": "relu", "residual": False, "f32": False},
        # the first MLP linear of a speech encoder's block (BASELINE config 1 with its activation), weights as the graph runtime leaves them
        {"name": "linear_fc1", "kind": "linear", "T": 1500, "K": 1280, "F": 5120, "layout": "kf", "epi": "gelu", "residual": False, "f32": False},
        # the same encoder's projection with the ragged extents the reference's census of declined GEMMs counts
        {"name": "linear_ragged", "kind": "linear", "T": 1544, "K": 1288, "F": 1288, "layout": "fk", "epi": "none", "residual": True, "f32": False},
        # global attention of a high-resolution image encoder
        {"name": "attention_global", "kind": "attention", "B": 1, "H": 16, "Lq": 4096, "Lk": 4096, "E": 64, "packed": False, "mask": "none", "f32": False},
        # windowed attention of such an encoder, head size 72, read in place from the packed projection; the last windows are padded
        {"name": "attention_windows", "kind": "attention", "B": 16, "H": 8, "Lq": 256, "Lk": 256, "E": 72, "packed": True, "mask": "pad", "f32": False},
        # the 3 x 3 convolution of the same encoder, channels first as exported graphs have it
        {"name": "conv_3x3", "kind": "conv", "N": 1, "Cin": 256, "Hi": 64, "Wi": 64, "Cout": 256, "k": 3, "s": 1, "p": 1, "act": "none"},
        # its patch stem: 7 x 7, stride 4, three input channels at full resolution
        {"name": "conv_stem", "kind": "conv", "N": 1, "Cin": 3, "Hi": 1024, "Wi": 1024, "Cout": 144, "k": 7, "s": 4, "p": 3, "act": "none"},
        # a mask decoder's upsampler: transposed convolution, kernel 2, stride 2
        {"name": "upsample_2x2", "kind": "upsample", "N": 1, "Cin": 256, "Hi": 64, "Wi": 64, "Cout": 64},
        # four blocks of a speech encoder over a 30 s window, captured once and replayed for every window
        {"name": "encoder_stack", "kind": "encoder", "T": 1500, "d": 1280, "layers": 4, "replay": True},
        # ViT-S/14 at 518 x 518 for one image after the other, captured and replayed
        {"name": "vit_518", "kind": "vit", "side": 518, "layers": 12, "replay": True},
        # a token of a speech decoder, batch 1: four layers over a full 448-slot cache and 1500 encoder states, then the
        # vocabulary; captured once, replayed per token
        {"name": "decode_token", "kind": "decode", "B": 1, "d": 1280, "layers": 4, "pos": 448, "src": 1500, "vocab": 51866, "replay": True},
        # a small ViT-S/14 from its exported graph over a batch of eight images, called as it is (no capture): host and GPU both count
        {"name": "exported_vit_b8", "kind": "exported", "B": 8, "side": 224, "layers": 12, "replay": False},
    ]


def _logint(rng, lo, hi):
    return int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))


def draw(rng):
    """One more case: any kind, sizes spread over its whole range on a logarithmic scale."""
    kind = rng.choices(["linear", "attention", "conv", "upsample", "encoder", "vit", "decode", "exported"], [5, 4, 3, 1, 2, 1, 3, 1])[0]
    while True:
        c = {"kind": kind}
        if kind == "linear":
            c.update(T=_logint(rng, 1, 8192), K=_logint(rng, 64, 5120), F=_logint(rng, 64, 8192))
            aligned = rng.random() < 0.75             # feature counts are mostly multiples of 64 or 8, sometimes anything (vocabularies, classes)
            if aligned:
                step = rng.choice([8, 64, 64])
                c.update(K=max(step, c["K"] // step * step), F=max(step, c["F"] // step * step))
            c.update(layout=rng.choice(["kf", "fk"]), epi=rng.choice(["none", "none", "gelu", "gelu_tanh", "relu"]), residual=rng.random() < 0.3)
            c.update(f32=not c["residual"] and rng.random() < 0.15)
            if work(c)["flops"] > (1.4e11 if aligned else 2e9):
                continue
        elif kind == "attention":
            same = rng.random() < 0.7
            Lk = _logint(rng, 16, 4096)
            c.update(B=_logint(rng, 1, 16), H=rng.choice([1, 2, 4, 6, 8, 12, 16, 20]), Lq=Lk if same else _logint(rng, 1, 4096), Lk=Lk,
                     E=rng.choice([16, 32, 64, 64, 64, 72, 128]), packed=same and rng.random() < 0.6, mask=rng.choice(["none", "none", "none", "pad", "dense"]),
                     f32=rng.random() < 0.15)
            if work(c)["flops"] > 7e10:
                continue
        elif kind == "conv":
            k, s = rng.choice([(1, 1), (3, 1), (3, 1), (3, 2), (5, 1), (7, 4)])
            c.update(N=rng.choice([1, 1, 2, 4]), Cin=rng.choice([3, 32, 64, 96, 128, 144, 256, 384]), Hi=_logint(rng, 8, 512), Wi=_logint(rng, 8, 512),
                     Cout=rng.choice([32, 64, 96, 144, 256, 384]), k=k, s=s, p=k // 2, act=rng.choice(["none", "relu"]))
            if work(c)["flops"] > 2e10:
                continue
        elif kind == "upsample":
            c.update(N=rng.choice([1, 1, 2]), Cin=rng.choice([32, 64, 96, 128, 256]), Hi=_logint(rng, 8, 160), Wi=_logint(rng, 8, 160),
                     Cout=rng.choice([16, 32, 48, 64, 128]))
        elif kind == "encoder":
            c.update(T=_logint(rng, 64, 1500), d=rng.choice([384, 512, 768, 1024, 1280]), layers=rng.randint(1, 4), replay=rng.random() < 0.6)
        elif kind == "vit":
            c.update(side=PATCH * rng.randint(8, 37), layers=rng.randint(2, 12), replay=rng.random() < 0.6)
        elif kind == "decode":
            c.update(B=rng.randint(1, 8), d=rng.choice([384, 512, 768, 1024, 1280]), layers=rng.randint(1, 4), pos=_logint(rng, 1, 448),
                     src=_logint(rng, 50, 1500), vocab=_logint(rng, 1000, 51866), replay=rng.random() < 0.6)
        else:
            c.update(B=rng.choice([1, 2, 4, 8]), side=PATCH * rng.randint(8, 37), layers=rng.randint(2, 12), replay=rng.random() < 0.4)
            if c["B"] * _vit_tokens(c["side"]) > 2800:
                continue
        return c


# ----------------------------------------------------------------------------- inputs

class _Draws:
    """Tensors of one seed, made on the GPU."""

    def __init__(self, seed):
        self.g = torch.Generator(device="cuda").manual_seed(int(seed))

    def randn(self, *shape, std=1.0, mean=0.0):
        t = torch.randn(shape, generator=self.g, device="cuda", dtype=torch.float32)
        return (t * std + mean).to(F16)

    def rand(self, *shape):
        return torch.rand(shape, generator=self.g, device="cuda", dtype=torch.float32).to(F16)

    def ints(self, hi, *shape):
        return torch.randint(0, hi, shape, generator=self.g, device="cuda")

    def weight(self, K, N, layout="kf", std=0.02):
        """A (K, N) linear weight in either memory layout."""
        return self.randn(K, N, std=std) if layout == "kf" else self.randn(N, K, std=std).t()

    def norm(self, n):
        return self.randn(n, std=0.02, mean=1.0), self.randn(n, std=0.02)


def _vit_tokens(side):
    return 1 + (side // PATCH) ** 2


def _linear(c, r):
    T, K, N = c["T"], c["K"], c["F"]
    s = {"x": r.randn(T, K), "w": r.weight(K, N, c["layout"], std=1.0 / math.sqrt(K)), "b": r.randn(N, std=0.02),
         "res": r.randn(T, N) if c["residual"] else None}
    s["out"] = torch.empty((T, N), dtype=torch.float32 if c["f32"] else F16, device="cuda")
    return s


def _run_linear(s):
    s["ctx"].ws.reset()
    return jv.matmul_(s["ctx"], s["out"], s["w"], s["x"], s["b"], epi=s["case"]["epi"], residual=s["res"])


def _attention(c, r):
    B, H, Lq, Lk, E = c["B"], c["H"], c["Lq"], c["Lk"], c["E"]
    heads = lambda t: t.unflatten(2, (H, E)).transpose(1, 2)                      # (B, L, H E) rows as the (B, H, L, E) operand
    if c["packed"]:                                                               # column bands of one projection
        qkv = r.randn(B, Lq, 3 * H * E)
        q, k, v = (heads(qkv[:, :, i * H * E:(i + 1) * H * E]) for i in range(3))
        out = heads(torch.empty((B, Lq, H * E), dtype=torch.float32 if c["f32"] else F16, device="cuda"))
    else:
        q, k, v = r.randn(B, H, Lq, E), r.randn(B, H, Lk, E), r.randn(B, H, Lk, E)
        out = torch.empty((B, H, Lq, E), dtype=torch.float32 if c["f32"] else F16, device="cuda")
    mask = None
    if c["mask"] == "pad":                                                        # key padding: each sequence with a length of its own
        length = Lk - r.ints(max(1, Lk // 3), B, 1)
        mask = torch.where(torch.arange(Lk, device="cuda")[None] < length, 0.0, torch.finfo(F16).min).to(F16).view(B, 1, 1, Lk)
    elif c["mask"] == "dense":                                                    # relative position bias, the same for the batch
        mask = r.randn(1, H, Lq, Lk)
    return {"q": q, "k": k, "v": v, "mask": mask, "out": out}


def _run_attention(s):
    s["ctx"].ws.reset()
    return jv.sdpa(s["ctx"], s["q"], s["k"], s["v"], s["mask"], out=s["out"])


def _conv_out(c):
    return tuple(jv.convsize(n, c["k"], c["s"], c["p"], 1) for n in (c["Hi"], c["Wi"]))


def _conv(c, r):
    k, OH, OW = c["k"], *_conv_out(c)
    return {"x": r.randn(c["N"], c["Cin"], c["Hi"], c["Wi"]), "w": r.randn(c["Cout"], c["Cin"], k, k, std=1.0 / math.sqrt(c["Cin"] * k * k)),
            "b": r.randn(c["Cout"], std=0.02), "out": torch.empty((c["N"], c["Cout"], OH, OW), dtype=F16, device="cuda")}


def _run_conv(s):
    c = s["case"]
    s["ctx"].ws.reset()
    return jv.convolution_(s["ctx"], s["out"], s["x"], s["w"], s["b"], (c["s"], c["s"]), (c["p"], c["p"]), (1, 1), 1, act=c["act"])


def _upsample(c, r):
    return {"x": r.randn(c["N"], c["Cin"], c["Hi"], c["Wi"]), "w": r.randn(c["Cin"], c["Cout"], 2, 2, std=1.0 / math.sqrt(c["Cin"])),
            "b": r.randn(c["Cout"], std=0.02), "out": torch.empty((c["N"], c["Cout"], 2 * c["Hi"], 2 * c["Wi"]), dtype=F16, device="cuda")}


def _run_upsample(s):
    s["ctx"].ws.reset()
    return jv.convolutiontranspose_(s["ctx"], s["out"], s["x"], s["w"], s["b"], (2, 2), (0, 0), (1, 1), (0, 0), 1)


def _layer(r, d, ffn, layout="kf"):
    w = lambda k, f: r.weight(k, f, layout)
    b = lambda n: r.randn(n, std=0.02)
    return EncoderLayerWeights(*r.norm(d), w(d, 3 * d), b(3 * d), w(d, d), b(d), *r.norm(d), w(d, ffn), b(ffn), w(ffn, d), b(d))


def _captured(s, step):
    """The step as the user's program runs it: itself, or its replay.  A captured graph holds addresses only, so the step
    is kept beside it: its closure owns the weights and buffers that the replays read and write."""
    s["eager"] = step
    s["step"] = StepGraph(step).replay if s["case"]["replay"] else step
    return s


def _run_step(s):
    s["step"]()
    return s["outs"]


def _encoder(c, r):
    T, d, n, ctx = c["T"], c["d"], c["layers"], jv.Ctx("cuda")
    folded = [fold_layer_norms(ctx, _layer(r, d, 4 * d)) for _ in range(n)]
    x, buf, st = r.randn(T, d), EncoderBuffers(T, d, 4 * d), FoldedStats(T, d)
    xs = [torch.empty((T, d), dtype=F16, device="cuda") for _ in range(2)]

    def step():
        src = x
        jv.rowstats_(ctx, st.x, x)
        for i, fw in enumerate(folded):
            encoder_layer_folded(ctx, fw, src, xs[i % 2], buf, st, d // 64, stats_out=i + 1 < n)
            src = xs[i % 2]
    return _captured({"case": c, "ctx": ctx, "x": x, "outs": xs[(n - 1) % 2]}, step)


def _vit(c, r):
    d, n, T, ctx = VIT_D, c["layers"], _vit_tokens(c["side"]), jv.Ctx("cuda")
    W = ViTWeights(r.randn(d, 3, PATCH, PATCH, std=0.02), r.randn(d, std=0.02), r.randn(1, d, std=0.02), r.randn(T, d, std=0.02),
                   [_layer(r, d, VIT_FFN) for _ in range(n)], *r.norm(d))
    enc = ViTEncoder(W, (c["side"], c["side"]), VIT_HEADS, VIT_FFN, fold_norms=ctx)
    image = r.rand(1, 3, c["side"], c["side"])
    return _captured({"case": c, "ctx": ctx, "x": image, "outs": enc.out}, lambda: enc(ctx, image))


def _decode(c, r):
    B, d, n, V, ctx = c["B"], c["d"], c["layers"], c["vocab"], jv.Ctx("cuda")
    w = lambda k, f: r.weight(k, f, "fk")                  # the layout decode-sized linears stream fastest (DecoderLayerWeights.k_contiguous)
    b = lambda m: r.randn(m, std=0.02)
    layers = [DecoderLayerWeights(*r.norm(d), w(d, 3 * d), b(3 * d), w(d, d), b(d), *r.norm(d), w(d, d), b(d), w(d, d), b(d), *r.norm(d),
                                  w(d, 4 * d), b(4 * d), w(4 * d, d), b(d)) for _ in range(n)]
    (g, beta), vocab = r.norm(d), w(d, V)
    cache = KVCache(n, B, d // 64, 64, src_len=c["src"])
    for t in (cache.self_k, cache.self_v, cache.cross_k, cache.cross_v):
        t.copy_(r.randn(*t.shape))
    cache.length.fill_(c["pos"])
    buf, xs = DecodeBuffers(B, d, 4 * d), [r.randn(B, d) for _ in range(n + 1)]
    h, logits = torch.empty((B, d), dtype=F16, device="cuda"), torch.empty((B, V), dtype=torch.float32, device="cuda")

    def step():
        cache.advance(ctx, 0)                              # the position stays where it is: every pass is the same token's work
        for i in range(n):
            decoder_layer_step(ctx, layers[i], cache, i, xs[i], xs[i + 1], buf)
        ctx.ws.reset()
        if B <= 4:
            jv.ln_matmul_(ctx, logits, vocab, xs[n], g, beta, 1e-5)
        else:
            jv.layernorm_(ctx, h, None, None, xs[n], g, beta, d, 1e-5)
            jv.matmul_(ctx, logits, vocab, h)
    return _captured({"case": c, "ctx": ctx, "outs": {"x": xs[n], "logits": logits, "k": cache.self_k, "v": cache.self_v}}, step)


class _Block(nn.Module):
    def __init__(self):
        super().__init__()
        d = VIT_D
        self.norm1, self.norm2 = nn.LayerNorm(d, eps=1e-6), nn.LayerNorm(d, eps=1e-6)
        self.qkv, self.proj, self.fc1, self.fc2 = nn.Linear(d, 3 * d), nn.Linear(d, d), nn.Linear(d, VIT_FFN), nn.Linear(VIT_FFN, d)
        self.ls1, self.ls2 = nn.Parameter(torch.ones(d)), nn.Parameter(torch.ones(d))

    def forward(self, x):
        B, N, C = x.shape
        E = C // VIT_HEADS
        qkv = self.qkv(self.norm1(x)).reshape(B, N, 3, VIT_HEADS, E).permute(2, 0, 3, 1, 4)
        a = F.scaled_dot_product_attention(qkv[0], qkv[1], qkv[2])
        x = x + self.proj(a.transpose(1, 2).reshape(B, N, C)) * self.ls1
        return x + self.fc2(F.gelu(self.fc1(self.norm2(x)))) * self.ls2


class _ViT(nn.Module):
    def __init__(self, side, layers):
        super().__init__()
        self.patch_embed = nn.Conv2d(3, VIT_D, PATCH, PATCH)
        self.cls_token, self.pos_embed = nn.Parameter(torch.empty(1, 1, VIT_D)), nn.Parameter(torch.empty(1, _vit_tokens(side), VIT_D))
        self.blocks = nn.ModuleList([_Block() for _ in range(layers)])
        self.norm = nn.LayerNorm(VIT_D, eps=1e-6)

    def forward(self, img):
        x = self.patch_embed(img).flatten(2).transpose(1, 2)
        x = torch.cat((self.cls_token.expand(x.shape[0], -1, -1), x), dim=1) + self.pos_embed
        for b in self.blocks:
            x = b(x)
        return self.norm(x)


@functools.lru_cache(maxsize=4)
def _exported_graph(B, side, layers):
    """The model's file, so to speak: its exported graph in the JSON schema, rewritten, and the shapes of its weights."""
    with torch.device("meta"):
        m = _ViT(side, layers).eval().half()
        table = torch.export.default_decompositions()
        table.pop(torch.ops.aten.scaled_dot_product_attention.default, None)
        ep = torch.export.export(m, (torch.empty(B, 3, side, side, dtype=F16),)).run_decompositions(table)
    return G.optimize(G.Graph.load(G.convert(ep, "vit"))), {k: tuple(v.shape) for k, v in m.state_dict().items()}


def _exported(c, r):
    graph, shapes = _exported_graph(c["B"], c["side"], c["layers"])
    mean = lambda k: 1.0 if (".norm" in k or k.startswith("norm.")) and k.endswith("weight") or ".ls" in k else 0.0
    weights = {k: r.randn(*shape, std=0.02, mean=mean(k)) for k, shape in sorted(shapes.items())}
    ctx = jv.Ctx("cuda")
    run, image = G.Executor(graph, weights, ctx), r.rand(c["B"], 3, c["side"], c["side"])
    if c["replay"]:
        replay, outs = run.replayable(image)
        return {"case": c, "ctx": ctx, "run": run, "step": replay, "outs": outs}
    return {"case": c, "ctx": ctx, "run": run, "x": image}


def _run_exported(s):
    return _run_step(s) if "step" in s else s["run"](s["x"])


_KINDS = {"linear": (_linear, _run_linear), "attention": (_attention, _run_attention), "conv": (_conv, _run_conv), "upsample": (_upsample, _run_upsample),
          "encoder": (_encoder, _run_step), "vit": (_vit, _run_step), "decode": (_decode, _run_step), "exported": (_exported, _run_exported)}


def prepare(case, seed):
    s = _KINDS[case["kind"]][0](case, _Draws(seed))
    s.setdefault("case", case)
    s.setdefault("ctx", None)
    if s["ctx"] is None:
        s["ctx"] = jv.Ctx("cuda")
    return s


def run(state):
    return _KINDS[state["case"]["kind"]][1](state)


# ----------------------------------------------------------------------------- what a pass cannot do without

def _encoder_work(T, d, ffn, n, images=1):
    """``n`` blocks over ``images`` sequences of ``T`` tokens: linears, attention; weights read once, activations in and out."""
    rows = T * images
    return {"flops": n * (2.0 * rows * d * (4 * d + 2 * ffn) + 4.0 * images * T * T * d), "bytes": 2.0 * (n * (4 * d * d + 2 * d * ffn) + 2 * rows * d)}


def work(case):
    c, kind = case, case["kind"]
    if kind == "linear":
        T, K, N = c["T"], c["K"], c["F"]
        return {"flops": 2.0 * T * K * N, "bytes": 2.0 * (T * K + K * N + N + (T * N if c["residual"] else 0)) + (4.0 if c["f32"] else 2.0) * T * N}
    if kind == "attention":
        n, mask = c["B"] * c["H"] * c["E"], {"none": 0, "pad": c["B"] * c["Lk"], "dense": c["H"] * c["Lq"] * c["Lk"]}[c["mask"]]
        return {"flops": 4.0 * n * c["Lq"] * c["Lk"], "bytes": 2.0 * (n * (c["Lq"] + 2 * c["Lk"]) + mask) + (4.0 if c["f32"] else 2.0) * n * c["Lq"]}
    if kind == "conv":
        OH, OW = _conv_out(c)
        crs = c["Cin"] * c["k"] ** 2
        return {"flops": 2.0 * c["N"] * OH * OW * crs * c["Cout"],
                "bytes": 2.0 * (c["N"] * (c["Cin"] * c["Hi"] * c["Wi"] + c["Cout"] * OH * OW) + crs * c["Cout"] + c["Cout"])}
    if kind == "upsample":
        px = c["N"] * c["Hi"] * c["Wi"]
        return {"flops": 8.0 * px * c["Cin"] * c["Cout"], "bytes": 2.0 * (px * (c["Cin"] + 4 * c["Cout"]) + 4 * c["Cin"] * c["Cout"] + c["Cout"])}
    if kind == "encoder":
        return _encoder_work(c["T"], c["d"], 4 * c["d"], c["layers"])
    if kind == "decode":
        B, d, n = c["B"], c["d"], c["layers"]
        weights, keys = n * 14.0 * d * d + d * c["vocab"], n * 2.0 * B * d * (c["pos"] + c["src"])
        return {"flops": 2.0 * B * weights + 2.0 * keys, "bytes": 2.0 * (weights + keys) + 4.0 * B * c["vocab"]}
    B, T = c.get("B", 1), _vit_tokens(c["side"])
    w, pixels = _encoder_work(T, VIT_D, VIT_FFN, c["layers"], B), B * 3.0 * c["side"] ** 2
    return {"flops": w["flops"] + 2.0 * B * (T - 1) * 3 * PATCH ** 2 * VIT_D, "bytes": w["bytes"] + 2.0 * (pixels + T * VIT_D + 3 * PATCH ** 2 * VIT_D)}


def tolerance(case):
    """What fp16 operands and results with fp32 sums leave open: the order of a sum moves a rounding of 2^-11 here and
    there.  Attention rounds its probabilities too; a stack of blocks carries such roundings through every layer."""
    kind = case["kind"]
    if kind == "linear":
        return {"rel": 1e-4 if case["f32"] else 1e-3}
    if kind in ("conv", "upsample"):
        return {"rel": 1e-3}
    if kind == "attention":
        return {"rel": 2e-3}
    return {"rel": 5e-3}
