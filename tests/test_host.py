"""What the native host side decides without a GPU: which memory a recorded call may move with an input."""
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
