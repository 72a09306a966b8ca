"""GPU parity of the large GEMMs through operand planes (k_plane.hip) with the
kernels that decode inside the K loop (k_nf4_bf16, oracle-tested): the
allocation-free backward always takes the latter, and planes take no call whose
reduction that kernel splits, so the input gradient's sums run in the same order
and the bits must match.  The forward is held against 64 bits on the dequantized weight.

The bar on the normalised error (parity.nerr) is 8 standard deviations of one
output's rounding error, as in tests/test_gpu_slim.py: 3.9e-6 for fp32 X (xl.wl and
the parts below hi + lo), 2.3e-6 for bf16 X (w below hi + lo, 0.18 x 2^-16 rms,
and the fp32 sums).
"""
import ctypes as C

import numpy as np
import pytest

import oracle as O
from parity import bf16_round, nerr

pytestmark = [pytest.mark.gpu, pytest.mark.timeout(120)]

torch = pytest.importorskip("torch")

TOL = {torch.float32: 8 * 4.8e-6, torch.bfloat16: 8 * 2.8e-6}


def _layer(QD, ctx, N, K, r, M, act, dq):
    g = O.Rng(N + 3 * K + 7 * M)
    dev = lambda v: torch.from_numpy(np.ascontiguousarray(v)).cuda()  # noqa: E731
    rnd = (lambda v: bf16_round(v)) if act == torch.bfloat16 else (lambda v: v)
    w, x = g.normal(N * K, 0.02).reshape(N, K), rnd(g.normal(M * K)).reshape(M, K)
    dy = rnd(g.normal(M * N)).reshape(M, N)
    a, b = g.uniform(r * K, -0.02, 0.02).reshape(r, K), g.normal(N * r, 0.01).reshape(N, r)
    W = QD.DeviceWeight.quantize(dev(w), 64, dq, ctx=ctx)
    ta, tb = dev(a), dev(b)
    return dict(W=W, wd=W.dequantize(ctx=ctx).view(N, K).double(), a=ta, b=tb, x=dev(x).to(act),
                dy=dev(dy).to(act), lora=QD.lora_struct(ta, tb, r, 16.0) if r else None,
                s=16.0 / r if r else 0.0, nx=x, ndy=dy)


def _backward(QD, ctx, fn, L, M):
    gx = torch.full((M, L["W"].cols), float("nan"), device="cuda")
    r = L["lora"].r if L["lora"] else 0
    ga, gb = (torch.empty(n, device="cuda") for n in (r * L["W"].cols or 1, r * L["W"].rows or 1))
    s = L["W"].struct()
    QD.check(fn(ctx.h, C.byref(s), C.byref(L["lora"]) if r else None, QD._p(L["x"]),
                QD._p(L["dy"]), QD._dt(L["x"]), M, None, QD._p(gx), QD._p(ga), QD._p(gb),
                C.c_void_p(torch.cuda.current_stream().cuda_stream)))
    return gx


CASES = [
    # (N, K, r, M): whole tiles; rows past a tile of 128, 192 and 256 rows;
    # columns past a tile; ranks around an MFMA's 16 and past four k tiles
    (4096, 2112, 16, 2048), (4352, 1088, 8, 1029), (8200, 1088, 64, 1900), (4200, 1088, 17, 1100),
    (4096, 1088, 16, 2905), (4104, 1088, 33, 3000), (4096, 1088, 0, 1100), (4104, 1088, 80, 1029),
    (2056, 2112, 5, 2900),
]


@pytest.mark.parametrize("act", [torch.float32, torch.bfloat16])
@pytest.mark.parametrize("N,K,r,M", CASES)
def test_plane_forward(ctx, N, K, r, M, act):
    from qlora_hip import device as QD
    for dq in (True, False):
        print(f"plane forward N={N} K={K} r={r} M={M} {act} dq={dq}", flush=True)
        L = _layer(QD, ctx, N, K, r, M, act, dq)
        y = torch.full((M, N), float("nan"), device="cuda")
        ctx.set_timing(True)
        QD.forward(L["W"], L["lora"], L["x"], M, y, ctx=ctx)
        torch.cuda.synchronize()
        rep = ctx.timing_report(reset=True)
        ctx.set_timing(False)
        assert "planes" in rep, rep
        xd = L["x"].double()
        want = xd @ L["wd"].T + L["s"] * ((xd @ L["a"].double().T) @ L["b"].double().T)
        assert nerr(y.cpu().numpy(), want.cpu().numpy(), K, L["nx"],
                    L["wd"].cpu().numpy()) < TOL[act]


@pytest.mark.parametrize("act", [torch.float32, torch.bfloat16])
@pytest.mark.parametrize("N,K,r,M", [(2056, 4096, 16, 2048), (1096, 4352, 8, 1029),
                                     (1096, 4096, 64, 2905), (1096, 4160, 5, 3000),
                                     (2056, 2112, 5, 2900)])
def test_plane_input_gradient(ctx, N, K, r, M, act):
    from qlora_hip import device as QD
    L = _layer(QD, ctx, N, K, r, M, act, True)
    ctx.set_timing(True)
    got = _backward(QD, ctx, ctx.lib.qh_qlora_backward_dev, L, M)
    torch.cuda.synchronize()
    rep = ctx.timing_report(reset=True)
    ctx.set_timing(False)
    assert "planes" in rep, rep
    ref = _backward(QD, ctx, ctx.lib.qh_qlora_backward_dev_noalloc, L, M)
    torch.cuda.synchronize()
    dy = L["dy"].double()
    want = dy @ L["wd"] + (L["s"] * (dy @ L["b"].double())) @ L["a"].double()
    for t in (got, ref):
        assert nerr(t.cpu().numpy(), want.cpu().numpy(), N, L["ndy"],
                    L["wd"].cpu().numpy()) < TOL[act]
    # both run dy.w (and its LoRA term) k by k in one chain
    assert torch.equal(got.view(torch.int32), ref.view(torch.int32))


@pytest.mark.parametrize("N,K,M", [
    (192, 576, 24000),     # few columns: a quarter of the products would be padding
    (33024, 2048, 100),    # few rows: writing the weight's planes costs more than the GEMM
    (4096, 512, 2048),     # a short reduction: two launches of 20 us each
])
def test_calls_that_planes_slow_down_stay_off_them(ctx, N, K, M):
    from qlora_hip import device as QD
    for act in (torch.float32, torch.bfloat16):
        W = QD.DeviceWeight.quantize(torch.randn(N, K, device="cuda") * 0.02, 64, True, ctx=ctx)
        Wt = QD.DeviceWeight.quantize(torch.randn(K, N, device="cuda") * 0.02, 64, True, ctx=ctx)
        x = torch.randn(M, K, device="cuda").to(act)
        ctx.set_timing(True)
        QD.forward(W, None, x, M, torch.empty(M, N, device="cuda"), ctx=ctx)
        fwd = ctx.timing_report(reset=True)
        QD.backward(Wt, None, torch.empty(M, N, device="cuda", dtype=act), x, M,
                    torch.empty(M, N, device="cuda"), ctx=ctx)
        torch.cuda.synchronize()
        bwd = ctx.timing_report(reset=True)
        ctx.set_timing(False)
        assert "planes" not in fwd and "planes" not in bwd, (fwd, bwd)


def test_codes_off_16_bytes_stay_off_planes(ctx):
    """k_nf4_bf16 reads codes 8 bytes at a time, the planes 16: a weight that
    starts on 8 bytes stays on the former, with the same bits."""
    from qlora_hip import device as QD
    N, K, M = 4096, 1088, 1100
    L = _layer(QD, ctx, N, K, 8, M, torch.float32, True)
    W, ys = L["W"], []
    for off in (0, 8):
        buf = torch.empty(W.codes.numel() + off, dtype=torch.uint8, device="cuda")
        buf[off:] = W.codes.reshape(-1)
        V = QD.DeviceWeight(N, K, 64, buf[off:], scale_codes=W.scale_codes, absmax=W.absmax)
        ys.append(torch.empty(M, N, device="cuda"))
        ctx.set_timing(True)
        QD.forward(V, L["lora"], L["x"], M, ys[-1], ctx=ctx)
        torch.cuda.synchronize()
        rep = ctx.timing_report(reset=True)
        ctx.set_timing(False)
        assert V.struct().codes % 16 == off and ("planes" in rep) == (off == 0), rep
    assert torch.equal(ys[0].view(torch.int32), ys[1].view(torch.int32))


@pytest.mark.parametrize("Ns,K,M,planes", [
    ((4352, 4352, 4352), 1088, 1024, (False, False)),  # one launch fills its rounds better
    ((2304, 2304, 2304), 2048, 2048, (False, False)),
    ((4096, 4096), 4096, 1100, (True, True)),
])
def test_groups_take_the_faster_of_planes_and_one_launch(ctx, Ns, K, M, planes):
    from qlora_hip import device as QD
    rnd = lambda *s: torch.randn(*s, device="cuda")  # noqa: E731
    Ls = [(QD.DeviceWeight.quantize(rnd(N, K) * 0.02, 64, True, ctx=ctx), None) for N in Ns]
    x, ys = rnd(M, K), [torch.empty(M, N, device="cuda") for N in Ns]
    dys, gx = [rnd(M, N) for N in Ns], torch.empty(M, K, device="cuda")
    ctx.set_timing(True)
    QD.forward_shared(Ls, x, M, ys, ctx=ctx)
    fwd = ctx.timing_report(reset=True)
    QD.backward_shared(Ls, x, dys, M, gx, ctx=ctx)
    torch.cuda.synchronize()
    bwd = ctx.timing_report(reset=True)
    ctx.set_timing(False)
    for rep, name, p in ((fwd, "forward_gemm_bf16", planes[0]), (bwd, "grad_x_gemm_bf16", planes[1])):
        assert ("planes" in rep) == p and rep[name][0] == (len(Ns) if p else 1), rep
    want = 0
    for (W, _), y, dy in zip(Ls, ys, dys):
        wd = W.dequantize(ctx=ctx).view(W.rows, K).double()
        w = x.double() @ wd.T
        assert float((y - w).norm() / w.norm()) < 2e-5
        want = want + dy.double() @ wd
    assert float((gx - want).norm() / want.norm()) < 2e-5


def test_plane_shared_sum(ctx):
    """Two layers that both take planes: the second adds its input gradient to
    the first's."""
    from qlora_hip import device as QD
    M, K = 1100, 4096
    Ls = [_layer(QD, ctx, N, K, 8, M, torch.float32, True) for N in (1088, 1152)]
    gx = torch.empty(M, K, device="cuda")
    ctx.set_timing(True)
    QD.backward_shared([(L["W"], L["lora"]) for L in Ls], Ls[0]["x"], [L["dy"] for L in Ls], M, gx,
                       [torch.empty(8, K, device="cuda") for _ in Ls],
                       [torch.empty(L["W"].rows, 8, device="cuda") for L in Ls], ctx=ctx)
    torch.cuda.synchronize()
    rep = ctx.timing_report(reset=True)
    ctx.set_timing(False)
    assert rep["planes"][0] == 2, rep
    want = sum(L["dy"].double() @ L["wd"] + (L["s"] * (L["dy"].double() @ L["b"].double())) @
               L["a"].double() for L in Ls)
    assert nerr(gx.cpu().numpy(), want.cpu().numpy(), 2240, Ls[0]["ndy"],
                Ls[0]["wd"].cpu().numpy()) < TOL[torch.float32]


def test_plane_residual(ctx):
    """The o projection of a block adds to x in the planes' GEMM; ragged rows."""
    from qlora_hip import device as QD
    M, h, r = 1100, 4096, 8
    L = _layer(QD, ctx, h, h, r, M, torch.float32, True)
    W = L["W"]
    blk = QD.AttnProjections(torch.ones(h, device="cuda"), W, W, W, W,
                             (None, None, None, (L["a"], L["b"], r, 16.0)), ctx=ctx)
    cache = blk.new_cache(M)
    cache["attn"].copy_(L["x"])
    x = torch.from_numpy(L["ndy"]).cuda()
    want = x.double()
    ctx.set_timing(True)
    blk.o_forward(x, cache)
    torch.cuda.synchronize()
    rep = ctx.timing_report(reset=True)
    ctx.set_timing(False)
    assert "planes" in rep and "residual_add" not in rep, rep
    xd = L["x"].double()
    want = want + xd @ L["wd"].T + L["s"] * ((xd @ L["a"].double().T) @ L["b"].double().T)
    assert nerr(x.cpu().numpy(), want.cpu().numpy(), h, L["nx"],
                L["wd"].cpu().numpy()) < TOL[torch.float32]


def test_plane_capture_without_warm_up(ctx):
    """A capture on a fresh context cannot have the planes' memory: the call takes
    the kernel that needs none, with the same bits; a warm context replays planes."""
    import qlora_hip as QH
    from qlora_hip import device as QD
    N, K, M = 4096, 1088, 1100
    L = _layer(QD, ctx, N, K, 0, M, torch.float32, True)
    y = torch.empty(M, N, device="cuda")
    QD.forward(L["W"], None, L["x"], M, y, ctx=ctx)
    torch.cuda.synchronize()
    want = y.clone()
    fresh = QH.Context()
    for c in (ctx, fresh):
        gr = torch.cuda.CUDAGraph()
        with torch.cuda.graph(gr):
            QD.forward(L["W"], None, L["x"], M, y, ctx=c)
        for _ in range(3):
            y.fill_(float("nan"))
            gr.replay()
            torch.cuda.synchronize()
            assert torch.equal(want.view(torch.int32), y.view(torch.int32))
        del gr
    fresh.close()
