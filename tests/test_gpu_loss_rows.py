"""Softmax cross-entropy rows whose start is off 16 bytes: every phase of the
row start against every remainder, from rows shorter than one vector to rows
past the register chunks (16 384 logits), with the target in the head, the
body and the tail.

Reference: the softmax in float64.  Bound per element: a value is one rounded
quotient of expf(v - max) (v - max exact to half an ulp of its size, at most
16 * 2^-24; expf a few ulp) and a sum of positive terms, whose error grows
with the length of the longest chain of additions (a thread's own chunk
values, then trees: under 256 here): 300 * 2^-24 = 1.8e-5 of the value, plus
the rounding of 1 / seq at the target.
"""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu

torch = pytest.importorskip("torch")


@pytest.mark.parametrize("inplace", [False, True])
@pytest.mark.parametrize("vocab", [1, 2, 3, 5, 6, 7, 9, 4095, 4097, 16383, 16385, 16386, 16387,
                                   16389, 65537, 131075])
def test_rows_off_sixteen_bytes(ctx, vocab, inplace):
    from qlora_hip import device as QD

    print("vocab", vocab, "inplace", inplace, flush=True)
    seq = 9
    rng = np.random.default_rng(vocab)
    x = (rng.standard_normal((seq, vocab)) * 2).astype(np.float32)
    tg = rng.integers(0, vocab, seq).astype(np.uint32)
    tg[:6] = [0, vocab - 1, min(1, vocab - 1), max(vocab - 2, 0), min(2, vocab - 1),
              max(vocab - 3, 0)]
    x64 = x.astype(np.float64)
    e = np.exp(x64 - x64.max(1, keepdims=True))
    p = e / e.sum(1, keepdims=True)
    want = p / seq
    want[np.arange(seq), tg] -= 1.0 / seq
    wloss = -np.mean(np.log(p[np.arange(seq), tg]))

    # guard values on both sides of the rows: nothing outside them is written
    buf = torch.full((seq * vocab + 8,), 7.0, device="cuda:0")
    out = buf[4:4 + seq * vocab].view(seq, vocab)
    src = torch.from_numpy(x).to("cuda:0")
    if inplace:
        out.copy_(src)
        src = out
    t = torch.from_numpy(tg.astype(np.int32)).to("cuda:0")
    loss, d = QD.softmax_cross_entropy(src, t, dlogits=out, ctx=ctx)
    got = d.cpu().numpy().astype(np.float64)
    assert torch.all(buf[:4] == 7.0) and torch.all(buf[4 + seq * vocab:] == 7.0)
    tol = 1.8e-5 * p / seq + 2.0 ** -23 / seq * (np.arange(vocab)[None, :] == tg[:, None])
    assert np.all(np.abs(got - want) <= tol + 1e-45)
    # the loss: terms of at most max|log p| with the same sum error, in fp32
    assert abs(float(loss) - wloss) <= 1.8e-5 + 2.0 ** -22 * abs(wloss)
