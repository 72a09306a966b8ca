"""GPU parity of the few-token forward (k_slim.hip: 17 tokens to some hundreds)
against the layer in 64 bits on the oracle's dequantized weight
(QloraLinear::forward, qlora-core/src/qlora.rs:86-107), at the edges of its
tiles: token groups of 16 and workgroups of 48 (fp32) or 64 (bf16) tokens, row
groups of 32 to 64, K of an odd number of blocks and of several
slices.

Bars on the normalised error (parity.nerr), 8 standard deviations of one
output's rounding error: an fp32 product drops xl.Ll and x's part below hi + lo,
each 0.18 x 2^-16 of it rms (a value uniform over its binade rounds to 8 bits
within 0.42 x 2^-8 rms, twice), together 3.9e-6; a bf16 product is exact up to
the codebook's 3.4e-7, the fp32 sums of some thousand terms add as much.
"""
import numpy as np
import pytest

import oracle as O
from parity import bf16_round, nerr

pytestmark = [pytest.mark.gpu, pytest.mark.timeout(120)]

torch = pytest.importorskip("torch")

TOL = {torch.float32: 8 * 3.9e-6, torch.bfloat16: 8 * 5e-7}
TOL_T1 = 2e-6  # fp32 products and sums: 8 x 2^-22 of an output's deviation


def _layer(QD, ctx, g, N, K, r, M, act, dq, x=None):
    w = g.normal(N * K, 0.02)
    a = g.uniform(r * K, -1 / np.sqrt(K), 1 / np.sqrt(K)).reshape(r, K)
    b = g.normal(N * r, 0.01).reshape(N, r)
    if x is None:
        x = g.normal(M * K).reshape(M, K)
        x = bf16_round(x) if act == torch.bfloat16 else x
    dev = lambda v: torch.from_numpy(np.ascontiguousarray(v)).cuda()  # noqa: E731
    W = QD.DeviceWeight.quantize(dev(w.reshape(N, K)), 64, dq, ctx=ctx)
    wd = O.dequantize(O.quantize(w, 64, dq)).reshape(N, K)
    ta, tb = dev(a), dev(b)
    lora = QD.lora_struct(ta, tb, r, 16.0) if r else None
    return dict(W=W, wd=wd, a=a, b=b, x=x, lora=lora, s=16.0 / r if r else 0.0,
                tx=dev(x).to(act), y=torch.full((M, N), float("nan"), device="cuda"),
                t1=torch.full((M, r), float("nan"), device="cuda") if r else None)


def _check(L, K, act):
    x = L["x"].astype(np.float64)
    want = x @ L["wd"].astype(np.float64).T
    if L["lora"] is not None:
        t1 = x @ L["a"].astype(np.float64).T
        want += L["s"] * (t1 @ L["b"].astype(np.float64).T)
        assert nerr(L["t1"].cpu().numpy(), t1, K, L["x"], L["a"]) < TOL_T1
    assert nerr(L["y"].cpu().numpy(), want, K, L["x"], L["wd"]) < TOL[act]


CASES = [
    # (N, K, r, M): tokens at the edges of a group and of a workgroup
    (96, 384, 16, 17), (96, 384, 16, 32), (96, 384, 16, 33), (96, 384, 16, 48),
    (96, 384, 16, 49), (96, 384, 16, 64), (96, 384, 16, 65), (96, 384, 16, 129),
    # K of an odd number of blocks (the last unit half empty)
    (40, 320, 8, 20), (72, 448, 4, 37), (130, 576, 8, 50), (64, 1088, 16, 24),
    # rows below and just past a row group; ranks of 1, 5, 16 + 1 and 64; none
    (1, 512, 1, 18), (33, 512, 5, 40), (65, 512, 17, 40), (127, 512, 64, 64), (64, 512, 0, 30),
    # several K slices (few rows, long K) with more than one token group
    (64, 8192, 16, 37), (16, 11008, 64, 60),
    # the largest token counts
    (256, 1024, 16, 512), (192, 576, 8, 384),
]


@pytest.mark.parametrize("act", [torch.float32, torch.bfloat16])
@pytest.mark.parametrize("N,K,r,M", CASES)
def test_slim_forward(ctx, N, K, r, M, act):
    from qlora_hip import device as QD
    for dq in (True, False):
        print(f"slim N={N} K={K} r={r} M={M} {act} dq={dq}", flush=True)
        L = _layer(QD, ctx, O.Rng(N * 7919 + K + M), N, K, r, M, act, dq)
        ctx.set_timing(True)
        QD.forward(L["W"], L["lora"], L["tx"], M, L["y"], t1=L["t1"], ctx=ctx)
        torch.cuda.synchronize()
        rep = ctx.timing_report(reset=True)
        ctx.set_timing(False)
        assert "forward_slim" in rep, rep
        _check(L, K, act)
        y0 = L["y"].clone()
        QD.forward(L["W"], L["lora"], L["tx"], M, L["y"], ctx=ctx)
        assert torch.equal(y0.view(torch.int32), L["y"].view(torch.int32))


WIDE = [
    # (N, K, r, M, dtypes): row groups of 48 and 64 rows (three and four 16-row
    # tiles a wave), each with every count of token groups that has them, rows
    # past a group; in the comment what slim_plan picks on 256 CUs
    (8243, 320, 33, 17, "fb"),    # 2 token groups, 3 tiles
    (12391, 320, 64, 17, "fb"),   # 2, 4
    (4101, 320, 64, 50, "f"),     # 2, 3 on two workgroups of tokens
    (6161, 320, 8, 49, "f"),      # 2, 4
    (2759, 576, 16, 100, "f"),    # 3, 3
    (4162, 320, 64, 70, "b"),     # 3, 3
    (6163, 576, 16, 70, "b"),     # 3, 4
    (4130, 576, 33, 100, "b"),    # 4, 3
    (9999, 1088, 64, 40, "fb"),   # 3, 3, two rounds
    (11008, 4096, 16, 37, "fb"),  # a 7B-class MLP's layer
]


@pytest.mark.parametrize("N,K,r,M,acts", WIDE)
def test_slim_wide_layers(ctx, N, K, r, M, acts):
    from qlora_hip import device as QD
    g = torch.Generator(device="cuda").manual_seed(N + K + M)
    rnd = lambda *s: torch.randn(*s, device="cuda", generator=g)  # noqa: E731
    w, a, b = rnd(N, K) * 0.02, rnd(r, K) / K ** 0.5, rnd(N, r) * 0.01
    lora = QD.lora_struct(a, b, r, 16.0)
    for act in [dict(f=torch.float32, b=torch.bfloat16)[c] for c in acts]:
        x = rnd(M, K).to(act)
        xd = x.double()
        t1w = xd @ a.double().T
        for dq in (True, False):
            print(f"slim wide N={N} K={K} r={r} M={M} {act} dq={dq}", flush=True)
            W = QD.DeviceWeight.quantize(w, 64, dq, ctx=ctx)
            wd = W.dequantize(ctx=ctx).view(N, K).double()
            y = torch.full((M, N), float("nan"), device="cuda")
            t1 = torch.full((M, r), float("nan"), device="cuda")
            ctx.set_timing(True)
            QD.forward(W, lora, x, M, y, t1=t1, ctx=ctx)
            torch.cuda.synchronize()
            rep = ctx.timing_report(reset=True)
            ctx.set_timing(False)
            assert "forward_slim" in rep, rep
            want = xd @ wd.T + (16.0 / r) * (t1w @ b.double().T)
            n = lambda t: t.cpu().numpy()  # noqa: E731
            assert nerr(n(t1), n(t1w), K, n(xd), n(a)) < TOL_T1
            assert nerr(n(y), n(want), K, n(xd), n(wd)) < TOL[act]


def test_slim_shared_layers_of_unequal_rows(ctx):
    """Four layers on one x in one launch: rows of 1 to 11 row groups, one
    without an adapter, K slices in all of them."""
    from qlora_hip import device as QD
    g, K, M = O.Rng(77), 4096, 41
    Ls, x = [], None
    for N, r in ((352, 16), (32, 0), (100, 64), (7, 3)):
        Ls.append(_layer(QD, ctx, g, N, K, r, M, torch.float32, True, x))
        x = Ls[0]["x"]
    QD.forward_shared([(L["W"], L["lora"]) for L in Ls], Ls[0]["tx"], M, [L["y"] for L in Ls],
                      t1s=[L["t1"] for L in Ls], ctx=ctx)
    torch.cuda.synchronize()
    for L in Ls:
        _check(L, K, torch.float32)


def test_slim_refused_forms_take_the_general_path(ctx):
    """A rank past 64, an x off 16 bytes, an in_dim off 64 and one below 320
    stay on the paths that took them before, with the same answer."""
    from qlora_hip import device as QD
    for N, K, r, off in ((64, 512, 65, 0), (64, 512, 8, 1), (64, 456, 8, 0), (64, 256, 8, 0)):
        L = _layer(QD, ctx, O.Rng(N + K + r), N, K, r, 40, torch.float32, True)
        if off:
            buf = torch.empty(40 * K + 1, device="cuda")
            buf[1:] = L["tx"].reshape(-1)
            L["tx"] = buf[1:].view(40, K)
        ctx.set_timing(True)
        QD.forward(L["W"], L["lora"], L["tx"], 40, L["y"], t1=L["t1"], ctx=ctx)
        torch.cuda.synchronize()
        rep = ctx.timing_report(reset=True)
        ctx.set_timing(False)
        assert "forward_slim" not in rep, rep
        x = L["x"].astype(np.float64)
        want = x @ L["wd"].astype(np.float64).T + L["s"] * (
            (x @ L["a"].astype(np.float64).T) @ L["b"].astype(np.float64).T)
        assert nerr(L["y"].cpu().numpy(), want, K, L["x"], L["wd"]) < 5e-5


@pytest.mark.parametrize("Ns,K,r,M", [
    ((136,), 2560, 0, 468),             # no adapter: the tiles are one short launch
    ((13904,), 768, 64, 126),           # rows enough to fill the tiles' one round
    ((1960, 1960, 640), 576, 0, 299),   # a group that the tiles run in one launch
    ((1752, 1752), 448, 8, 300),
])
def test_calls_that_slim_slows_down_stay_on_the_tiles(ctx, Ns, K, r, M):
    from qlora_hip import device as QD
    for act in (torch.float32, torch.bfloat16):
        Ls, x = [], None
        for N in Ns:
            Ls.append(_layer(QD, ctx, O.Rng(N + K), N, K, r, M, act, True, x))
            x = Ls[0]["x"]
        ctx.set_timing(True)
        if len(Ns) == 1:
            QD.forward(Ls[0]["W"], Ls[0]["lora"], Ls[0]["tx"], M, Ls[0]["y"], ctx=ctx)
        else:
            QD.forward_shared([(L["W"], L["lora"]) for L in Ls], Ls[0]["tx"], M,
                              [L["y"] for L in Ls], ctx=ctx)
        torch.cuda.synchronize()
        rep = ctx.timing_report(reset=True)
        ctx.set_timing(False)
        assert "forward_slim" not in rep, rep


def test_slim_under_capture(ctx):
    """A captured forward replays to the eager bits; so does one on a context
    whose scratch would have to grow, where a path that needs none takes it."""
    from qlora_hip import device as QD
    import qlora_hip as QH
    L = _layer(QD, ctx, O.Rng(5), 1152, 320, 0, 40, torch.float32, True)
    QD.forward(L["W"], None, L["tx"], 40, L["y"], ctx=ctx)
    torch.cuda.synchronize()
    want = L["y"].clone()
    fresh = QH.Context()
    for c, same in ((ctx, True), (fresh, False)):
        L["y"].fill_(float("nan"))
        gr = torch.cuda.CUDAGraph()
        with torch.cuda.graph(gr):
            QD.forward(L["W"], None, L["tx"], 40, L["y"], ctx=c)
        for _ in range(3):
            L["y"].fill_(float("nan"))
            gr.replay()
            torch.cuda.synchronize()
            if same:
                assert torch.equal(want.view(torch.int32), L["y"].view(torch.int32))
            else:
                _check(L, 320, torch.float32)
    del gr
    fresh.close()
