"""What the native host side decides without a GPU: which memory a recorded call may move with an input, what becomes of an
operand that torch refuses to look into."""
import subprocess
import sys

import torch

from juliavision_amd import kernels as K


def test_memory_that_two_tensors_share_is_not_apart():
    buf = torch.zeros(64, dtype=torch.float16)
    a, b, c = buf[:16], buf[16:32], buf[8:24]
    columns = buf.view(8, 8)[:, :4], buf.view(8, 8)[:, 4:]                       # interleaved: their spans overlap
    spans = lambda *ts: [K.span(t) for t in ts]
    assert K.span(columns[1]) == (buf.data_ptr() + 8, 2 * (7 * 8 + 4))
    assert K.apart(spans(a, b), []) and K.apart(spans(a), spans(b)) and K.apart([], spans(a, c))
    assert not K.apart(spans(a, c), []) and not K.apart(spans(b, a), spans(c)) and not K.apart(spans(*columns), [])
    assert not K.apart(spans(a), spans(buf)) and not K.apart(spans(buf), spans(b))      # one inside the other, either way round
    assert K.apart(spans(a, buf[:0]), spans(buf[4:4]))                            # nothing shares memory with an empty tensor


REFUSED = """
import torch
from torch._subclasses.fake_tensor import FakeTensorMode
from juliavision_amd import _lib as L, kernels as K
host = L.load_host()
host.setup(K.Workspace, K.Ctx)
ctx = object.__new__(K.Ctx)
ctx.dev = ctx._own = K.MI355X
ctx.device, ctx.ws = torch.device("cuda"), None
with FakeTensorMode():                                  # tensors that say "cuda" and have no storage, on a machine without the device
    h = lambda *s: torch.empty(s, dtype=torch.float16, device="cuda")
    f = lambda *s: torch.empty(s, dtype=torch.float32, device="cuda")
    x, q, i = h(16, 64), h(1, 2, 16, 64), h(1, 8, 8, 8)
    length = torch.empty(1, dtype=torch.int32, device="cuda")
    print(host.add(ctx, x, x, x), host.layernorm(ctx, x, x, None, None, 64, 1e-5), host.rowstats(ctx, f(2, 16, 2), x),
          host.matmul(ctx, x, h(64, 64), x, None, "none", None), host.matmul_rowstats(ctx, x, f(2, 16, 2), h(64, 64), x, None, "none", None, None),
          host.lnfold_matmul(ctx, x, h(64, 64), f(64), f(64), 1, x, f(2, 16, 2), 1e-5, "none", None, None, None),
          host.ln_matmul(ctx, h(4, 64), h(64, 64), h(4, 64), None, None, 1e-5, None, "none", None),
          host.sdpa(ctx, q, q, q, None, None, q, None),
          host.sdpa_append(ctx, h(1, 2, 1, 64), q, q, h(1, 2, 1, 64), h(1, 2, 1, 64), length, None, h(1, 2, 1, 64)),
          host.convolution(ctx, i, i, h(8, 8, 3, 3), None, (1, 1), (1, 1), (1, 1), 1, "none"),
          host.convolutiontranspose(ctx, h(1, 4, 16, 16), i, h(8, 4, 2, 2), None, (2, 2), (0, 0), (1, 1), (0, 0), 1),
          host.calls_run(ctx, host.calls_new([], []), (x,)))
"""


def test_what_torch_throws_sends_the_call_to_python():
    """An operand without storage or a device that is gone: the native functions answer False, and the Python forms raise."""
    r = subprocess.run([sys.executable, "-c", REFUSED], capture_output=True, text=True, timeout=300)
    assert r.returncode == 0, (r.returncode, r.stderr[-2000:])
    assert r.stdout.split() == ["False"] * 12
