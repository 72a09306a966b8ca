"""GPU parity of k_nf4_bf16's large tiles (256 x 256 and 256 x 128) against 64 bits,
in calls that do not take operand planes: a forward over a short reduction, and
the input gradient of the allocation-free backward.  Bar as in
tests/test_gpu_plane.py (the same sums)."""
import pytest

from parity import nerr
from test_gpu_plane import TOL, _backward

pytestmark = [pytest.mark.gpu, pytest.mark.timeout(120)]

torch = pytest.importorskip("torch")

R = 16


def _layer(QD, ctx, N, K, M, act):
    g = torch.Generator(device="cuda").manual_seed(N + 3 * K + M)
    rnd = lambda *s: torch.randn(*s, device="cuda", generator=g)  # noqa: E731
    a, b, x, dy = rnd(R, K) * 0.02, rnd(N, R) * 0.01, rnd(M, K).to(act), rnd(M, N).to(act)
    W = QD.DeviceWeight.quantize(rnd(N, K) * 0.02, 64, True, ctx=ctx)
    return dict(W=W, wd=W.dequantize(ctx=ctx).view(N, K).double(), a=a.double(), b=b.double(),
                x=x, dy=dy, lora=QD.lora_struct(a, b, R, 16.0))


@pytest.mark.parametrize("act", [torch.float32, torch.bfloat16])
@pytest.mark.parametrize("N,K,M", [
    (7900, 320, 4000),   # 16 x 31 tiles of 256 x 256, the last ones ragged
    (4200, 320, 4100),   # 17 x 33 tiles of 256 x 128
])
def test_large_tile_forward(ctx, N, K, M, act):
    from qlora_hip import device as QD
    L = _layer(QD, ctx, N, K, M, act)
    y = torch.full((M, N), float("nan"), device="cuda")
    ctx.set_timing(True)
    QD.forward(L["W"], L["lora"], L["x"], M, y, ctx=ctx)
    torch.cuda.synchronize()
    rep = ctx.timing_report(reset=True)
    ctx.set_timing(False)
    assert "forward_gemm_bf16" in rep and "planes" not in rep, rep
    x = L["x"].double()
    want = x @ L["wd"].T + (x @ L["a"].T) @ L["b"].T
    assert nerr(y.cpu().numpy(), want.cpu().numpy(), K, x.cpu().numpy(),
                L["wd"].cpu().numpy()) < TOL[act]


@pytest.mark.parametrize("act", [torch.float32, torch.bfloat16])
@pytest.mark.parametrize("N,K,M", [(520, 7872, 4000), (520, 4160, 4100)])
def test_large_tile_input_gradient(ctx, N, K, M, act):
    from qlora_hip import device as QD
    L = _layer(QD, ctx, N, K, M, act)
    got = _backward(QD, ctx, ctx.lib.qh_qlora_backward_dev_noalloc, L, M)
    torch.cuda.synchronize()
    dy = L["dy"].double()
    want = dy @ L["wd"] + (dy @ L["b"]) @ L["a"]
    assert nerr(got.cpu().numpy(), want.cpu().numpy(), N, dy.cpu().numpy(),
                L["wd"].cpu().numpy()) < TOL[act]
