"""Captured calls on a context whose scratch other calls grow: a graph keeps
the memory it was captured with (csrc/dev_buf.h; tests/test_dev_buf.py shows on
the CPU that the block stays owned), so a replay after a larger eager call
gives the bits of the eager call it stands for."""
import pytest

pytestmark = [pytest.mark.gpu, pytest.mark.timeout(120)]

torch = pytest.importorskip("torch")


def _layer(QD, ctx, N, K, r):
    g = torch.Generator(device="cuda").manual_seed(N + K + r)
    rnd = lambda *s: torch.randn(*s, device="cuda", generator=g)  # noqa: E731
    W = QD.DeviceWeight.quantize(rnd(N, K) * 0.02, 64, True, ctx=ctx)
    return W, QD.lora_struct(rnd(r, K) * 0.02, rnd(N, r) * 0.01, r, 16.0) if r else None


def _bits(t):
    return t.view(torch.int32)


def _capture(step):
    gr = torch.cuda.CUDAGraph()
    with torch.cuda.graph(gr):
        step()
    return gr


@pytest.mark.parametrize("M", [4, 37])  # the split decode kernel, the few-token forward
def test_replay_after_a_larger_eager_call(M):
    import qlora_hip as QH
    from qlora_hip import device as QD
    c = QH.Context()
    W, lora = _layer(QD, c, 11008, 4096, 16)
    x = torch.randn(2048, 4096, device="cuda")
    y, big = torch.empty(M, 11008, device="cuda"), torch.empty(2048, 11008, device="cuda")
    step = lambda: QD.forward(W, lora, x[:M], M, y, ctx=c)  # noqa: E731
    step()
    torch.cuda.synchronize()
    want = y.clone()
    gr = _capture(step)
    for _ in range(3):
        QD.forward(W, lora, x, 2048, big, ctx=c)  # needs more memory than the graph's call
        torch.cuda.synchronize()
        y.fill_(float("nan"))
        gr.replay()
        torch.cuda.synchronize()
        assert torch.equal(_bits(want), _bits(y))
    del gr
    c.close()


def test_capture_of_fewer_tokens_than_warmed_up():
    """The few-token kernel splits K at 33 tokens of this layer and not at 49, so
    its scratch for 33 exceeds that for 49; the tiles' does not."""
    import qlora_hip as QH
    from qlora_hip import device as QD
    c, d = QH.Context(), QH.Context()
    W, lora = _layer(QD, c, 2048, 4096, 8)
    x = torch.randn(49, 4096, device="cuda")
    y, want = torch.empty(49, 2048, device="cuda"), torch.empty(33, 2048, device="cuda")
    QD.forward(W, lora, x, 49, y, ctx=c)
    QD.forward(W, lora, x[:33], 33, want, ctx=d)
    torch.cuda.synchronize()
    gr = _capture(lambda: QD.forward(W, lora, x[:33], 33, y, ctx=c))
    for _ in range(3):
        y.fill_(float("nan"))
        gr.replay()
        torch.cuda.synchronize()
        # two splits of fp32 products into bf16 parts, 5e-6 of the norm each
        assert float((y[:33] - want).norm() / want.norm()) < 2e-5
    del gr
    c.close(), d.close()
