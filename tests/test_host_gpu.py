"""The native host side: an exported graph's recorded calls issued again on other inputs, and the calls it leaves to Python."""
import pytest
import torch
import torch.nn as nn
import torch.nn.functional as F

pytestmark = pytest.mark.gpu


class _Net(nn.Module):
    def __init__(self, d, heads):
        super().__init__()
        self.heads, self.norm = heads, nn.LayerNorm(d)
        self.q, self.k, self.v, self.o, self.fc = (nn.Linear(d, d) for _ in range(5))

    def attended(self, x):
        B, T, D = x.shape
        split = lambda t: t.view(B, T, self.heads, D // self.heads).transpose(1, 2)
        y = self.norm(x)
        a = F.scaled_dot_product_attention(split(self.q(y)), split(self.k(y)), split(self.v(y)))
        return x + self.o(a.transpose(1, 2).reshape(B, T, D))

    def forward(self, x):
        return self.attended(x), F.gelu(self.fc(x))


class _State(_Net):
    """One result, of the input's shape; its last op reads the input elementwise, so it may be handed back."""

    def forward(self, x):
        return self.attended(x)


@pytest.mark.parametrize("T", [5, 130])
def test_recorded_calls_follow_their_inputs(T):
    import juliavision_amd as jv
    from juliavision_amd import graph as G
    torch.manual_seed(T)
    m = _Net(128, 2).eval().half()
    g = G.optimize(G.Graph.load(G.convert(torch.export.export(m, (torch.randn(1, T, 128).half(),)), "net")))
    run = G.Executor(g, m.state_dict(), jv.Ctx("cuda"))
    xs = [torch.randn(1, T, 128, device="cuda").half() for _ in range(5)]
    shifted = torch.randn(8 + T * 128, device="cuda").half()[8:].view(1, T, 128)      # another alignment: not the calls recorded for xs
    for i, x in enumerate(xs[:3] + [shifted, shifted] + xs[3:]):
        got = [t.float().clone() for t in run(x)]
        if i == 4:
            run.ctx.ws.scratch(4 * run.ctx.ws.buf.numel())                                 # the workspace moves: recorded addresses are stale
        fresh = G.Executor(g, m.state_dict(), jv.Ctx("cuda"))(x)
        for a, b in zip(got, fresh):
            assert torch.equal(a, b.float()), f"run {i}"
    assert run._calls is not None


@pytest.mark.parametrize("T", [5, 130])
def test_a_result_handed_back_is_not_taken_for_an_input(T):
    """``x = run(x)``: the run that is noted must not take the result buffer for an input's memory, or the next call on a tensor
    of the user's writes its result there."""
    import juliavision_amd as jv
    from juliavision_amd import graph as G
    torch.manual_seed(T)
    m = _State(128, 2).eval().half()
    g = G.optimize(G.Graph.load(G.convert(torch.export.export(m, (torch.randn(1, T, 128).half(),)), "state")))
    run, ref = (G.Executor(g, m.state_dict(), jv.Ctx("cuda")) for _ in range(2))
    x = torch.randn(1, T, 128, device="cuda").half()
    want = x
    for i in range(4):
        want = ref(want.clone()).clone()
        x = run(x)
        assert torch.equal(x, want), f"pass {i}"
    for i in range(4):
        z = torch.randn(1, T, 128, device="cuda").half()
        kept = z.clone()
        got = run(z)
        assert torch.equal(z, kept), f"the input of call {i} was written to"
        assert torch.equal(got, G.Executor(g, m.state_dict(), jv.Ctx("cuda"))(kept)), f"call {i}"
    assert run._calls is not None


class _Two(nn.Module):
    def __init__(self, d):
        super().__init__()
        self.a, self.b = nn.Linear(d, d), nn.Linear(d, d)

    def forward(self, x, y):
        return self.a(x) + self.b(y)


@pytest.mark.parametrize("why", ["shared", "refused", "described"])
def test_calls_that_are_not_noted_are_not_noted_again(why, monkeypatch):
    """Inputs that share memory, a call that cannot be repeated, a context that the native side does not take: the runs that
    follow go through the handlers and their native calls, not through the recorder's slow ones."""
    import juliavision_amd as jv
    from juliavision_amd import graph as G, kernels as K
    torch.manual_seed(0)
    m, T = _Two(64).eval().half(), 20
    g = G.optimize(G.Graph.load(G.convert(torch.export.export(m, (torch.randn(T, 64).half(),) * 2), "two")))
    run, made = G.Executor(g, m.state_dict(), jv.Ctx("cuda", dev=jv.MI355X if why == "described" else None)), []

    class Recorder(K.CallRecorder):
        def __init__(self, ctx):
            made.append(self)
            super().__init__(ctx)

        def calls(self, inputs):
            return None if why == "refused" else super().calls(inputs)
    monkeypatch.setattr(K, "CallRecorder", Recorder)
    x, y = (torch.randn(T, 64, device="cuda").half() for _ in range(2))
    for i in range(5):
        args = (x, x) if why == "shared" else (x, y)
        got = run(*args)
        assert torch.equal(got, G.Executor(g, m.state_dict(), jv.Ctx("cuda"))(*args)), f"run {i}"
    assert len(made) == (why != "shared") and (run._calls is not None) == (why == "described")
    if why == "shared":                                                               # ... and apart again they are noted
        for _ in range(2):
            run(x, y)
        assert run._calls is not None and len(made) == 1


def test_a_subclass_of_the_context_keeps_its_stream():
    import juliavision_amd as jv
    side = torch.cuda.Stream()
    asked = []

    class Mine(jv.Ctx):
        @property
        def stream(self):
            asked.append(1)
            return side.cuda_stream
    ctx = Mine("cuda")
    x = torch.randn(16, 64, device="cuda").half()
    side.wait_stream(torch.cuda.current_stream())
    out = jv.add_(ctx, torch.empty_like(x), x, x)
    torch.cuda.synchronize()
    assert asked and torch.equal(out, x + x)


def test_threads_issue_calls_at_once():
    import threading
    import juliavision_amd as jv
    torch.manual_seed(0)
    w, xs = torch.randn(256, 512, device="cuda").half(), [torch.randn(40, 256, device="cuda").half() for _ in range(4)]
    want = [jv.matmul_(jv.Ctx("cuda"), torch.empty(40, 512, dtype=torch.float16, device="cuda"), w, x).clone() for x in xs]
    bad = []

    def work(i):
        ctx, out = jv.Ctx("cuda"), torch.empty(40, 512, dtype=torch.float16, device="cuda")
        for _ in range(50):
            ctx.ws.reset()
            jv.matmul_(ctx, out, w, xs[i])
        torch.cuda.synchronize()
        if not torch.equal(out, want[i]):
            bad.append(i)
    threads = [threading.Thread(target=work, args=(i,)) for i in range(4)]
    for t in threads:
        t.start()
    for t in threads:
        t.join()
    assert not bad


def test_what_the_native_side_leaves_is_still_refused_by_name():
    import juliavision_amd as jv
    ctx = jv.Ctx("cuda")
    h = lambda *s: torch.zeros(s, dtype=torch.float16, device="cuda")
    with pytest.raises(jv.DeclineError, match="bias"):
        jv.matmul_(ctx, h(16, 64), h(64, 64), h(16, 64), torch.zeros(64, device="cuda"))
    with pytest.raises(jv.DeclineError, match="extent"):
        jv.matmul_(ctx, h(16, 64), h(64, 64), h(16, 32))
    with pytest.raises(jv.DeclineError, match="residual"):
        jv.matmul_(ctx, h(16, 64), h(64, 64), h(16, 64), residual=h(16, 32))
    with pytest.raises(jv.DeclineError, match="nocoopmat"):
        jv.matmul_(jv.Ctx("cuda", dev=jv.MI355X._replace(coopmat=False)), h(16, 64), h(64, 64), h(16, 64))
    with pytest.raises(jv.DeclineError, match="extent"):
        jv.sdpa(ctx, h(1, 2, 8, 64), h(1, 2, 9, 64), h(1, 2, 8, 64), out=h(1, 2, 8, 64))
    torch.cuda.synchronize()
