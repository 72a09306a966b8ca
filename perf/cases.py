"""The workloads whose speed this repository is judged by, through its public
entry points (``qlora_hip`` and ``qlora_hip.device``).

``listed()`` names them; ``draw(rng)`` gives more of the same ranges.  A case
is a dict of plain values; its ``kind`` is one of

  layer     one QLoRA projection: forward, or forward and backward
  decode    a decode loop's captured graph over independent projections
  block     a decoder block's projections around the caller's attention
            (norm, q/k/v, o, MLP): forward, or forward and backward
  quantize  a float32 weight into packed NF4
  adam      the 8-bit Adam step over the adapters of some layers
  loss      softmax cross-entropy with its gradient

Weights are packed in plain torch from normal draws, as a program that loads a
packed checkpoint holds them, so that ``exact`` knows them bit for bit.
"""
import ctypes as C
import math
import os
import sys

import torch

sys.path.insert(0, os.path.join(os.getcwd(), "vkqlora.rs_amd"))

import qlora_hip as QH  # noqa: E402
from qlora_hip import device as QD  # noqa: E402

DEV = "cuda:0"
LEVELS = (-1.0, -0.6961928009986877, -0.5250730514526367, -0.39491748809814453,
          -0.28444138169288635, -0.18477343022823334, -0.09105003625154495, 0.0,
          0.07958029955625534, 0.16093020141124725, 0.24611230194568634,
          0.33791524171829224, 0.44070982933044434, 0.5626170039176941,
          0.7229568362236023, 1.0)
EPS = 1e-5


# ---- the cases ---------------------------------------------------------------
def listed():
    return [
        # one small layer of a 576-wide model, 64 tokens: seven short kernels,
        # where launches and latency count
        dict(name="tiny_layer", kind="layer", out=576, inp=576, tokens=64, r=8, act="f32",
             dq=True, train=True),
        # one token through the MLP projections of four 7B-class layers: the
        # latency of a single user's decode step
        dict(name="decode_7b_b1", kind="decode", out=11008, inp=4096, pairs=4, batch=1, r=16,
             act="f32", dq=True),
        # the same layers for sixteen users at once
        dict(name="decode_7b_b16", kind="decode", out=11008, inp=4096, pairs=4, batch=16, r=16,
             act="f32", dq=True),
        # a 70B-class MLP's projections for four users, bf16 activations
        dict(name="decode_70b_b4", kind="decode", out=28672, inp=8192, pairs=1, batch=4, r=64,
             act="bf16", dq=True),
        # a 7B-class block over a ragged serving batch: a short prompt, or
        # some tens of users a step
        dict(name="serve_block_37", kind="block", hidden=4096, kv=4096, inter=11008, seq=37,
             r=16, train=False),
        # training, one 4096 x 4096 projection, fp32 activations
        dict(name="train_4096_f32", kind="layer", out=4096, inp=4096, tokens=4096, r=64,
             act="f32", dq=True, train=True),
        # training, a wide projection in bf16 over a ragged packed batch,
        # weight scales not double-quantized
        dict(name="train_14336_bf16", kind="layer", out=14336, inp=4096, tokens=2905, r=64,
             act="bf16", dq=False, train=True),
        # training, one block of a 135M model (9 query and 3 key/value heads)
        dict(name="train_smol_block", kind="block", hidden=576, kv=192, inter=1536, seq=2048,
             r=8, train=True),
        # training, one block of a 70B-class model (8 key/value heads)
        dict(name="train_70b_block", kind="block", hidden=8192, kv=1024, inter=28672, seq=2048,
             r=64, train=True),
        # preparing a 70B-class weight
        dict(name="quantize_70b", kind="quantize", out=28672, inp=8192, dq=True),
        # the optimizer step over two 70B-class layers' adapters
        dict(name="adam_70b", kind="adam", out=28672, inp=8192, r=64, layers=1, pages=0),
        # the loss of a 2048-token batch over a 128k vocabulary
        dict(name="loss_128k", kind="loss", seq=2048, vocab=128256),
    ]


def _log(rng, lo, hi, step=1):
    """An integer from lo to hi, evenly over its logarithm, a multiple of step."""
    v = math.exp(rng.uniform(math.log(lo), math.log(hi)))
    return max(lo, min(hi, int(round(v / step)) * step))


def draw(rng):
    kind = rng.choice(["layer"] * 4 + ["decode"] * 3 + ["block"] * 3 +
                      ["quantize", "adam", "loss"])
    act = rng.choice(["f32", "bf16"])
    r = rng.choice([4, 8, 16, 32, 64])
    dq = rng.random() < 0.75
    if kind == "layer":
        # model widths are multiples of 64; output counts of 8
        return dict(kind=kind, out=_log(rng, 192, 14336, 8), inp=_log(rng, 192, 14336, 64),
                    tokens=_log(rng, 17, 4096), r=r, act=act, dq=dq, train=rng.random() < 0.6)
    if kind == "decode":
        out, inp = _log(rng, 1024, 28672, 256), _log(rng, 1024, 8192, 256)
        pairs = max(1, min(8, int(2.0e8 / (out * inp))))
        return dict(kind=kind, out=out, inp=inp, pairs=pairs, batch=_log(rng, 1, 16), r=r,
                    act=act, dq=dq)
    if kind == "block":
        hidden = _log(rng, 576, 5120, 64)
        kv = max(64, hidden // rng.choice([1, 3, 4, 8]) // 64 * 64)
        return dict(kind=kind, hidden=hidden, kv=kv,
                    inter=_log(rng, 2 * hidden, 4 * hidden, 64), seq=_log(rng, 17, 2048), r=r,
                    train=rng.random() < 0.6)
    if kind == "quantize":
        return dict(kind=kind, out=_log(rng, 192, 28672, 8), inp=_log(rng, 192, 8192, 64), dq=dq)
    if kind == "adam":
        return dict(kind=kind, out=_log(rng, 192, 14336, 8), inp=_log(rng, 192, 8192, 64), r=r,
                    layers=rng.randint(1, 16), pages=rng.choice([0, 4]))
    return dict(kind=kind, seq=_log(rng, 33, 2048), vocab=_log(rng, 8192, 131072))


# ---- inputs (plain torch, from the seed alone) ----------------------------------
def _gen(seed):
    return torch.Generator(device=DEV).manual_seed(seed)


def _randn(g, *shape, std=1.0):
    return torch.randn(*shape, device=DEV, generator=g).mul_(std)


def _packed(g, out, inp, dq):
    """A packed NF4 weight of W ~ 0.02 N(0, 1) in 64-element blocks: codes
    (element 2i in the low nibble), and int8 scale codes with one absmax per
    256 blocks, or fp32 scales."""
    w = _randn(g, out * inp // 64, 64, std=0.02)
    s = w.abs().amax(1)
    lv = torch.tensor(LEVELS, device=DEV)
    c = torch.bucketize(w / s[:, None], (lv[1:] + lv[:-1]) / 2, out_int32=True).to(torch.uint8)
    del w
    c = c.view(-1, 2)
    p = dict(rows=out, cols=inp, codes=c[:, 0] | (c[:, 1] << 4))
    if not dq:
        p["scales"] = s
        return p
    nb = s.numel()
    groups = torch.nn.functional.pad(s, (0, -nb % 256)).view(-1, 256)
    am = groups.amax(1)
    sc = (groups / am[:, None] * 127).round().view(-1)[:nb]
    p["scale_codes"], p["absmax"] = sc.to(torch.uint8), am  # 0 .. 127
    return p


def _weight(p):
    return QD.DeviceWeight(p["rows"], p["cols"], 64, p["codes"], p.get("scales"),
                           p.get("scale_codes"), p.get("absmax"))


def _dense(p):
    """The packed weight's values (the format defines them in fp32) in 64 bits."""
    lv = torch.tensor(LEVELS, device=DEV)
    c = torch.stack([p["codes"] & 15, p["codes"] >> 4], 1).view(-1, 64)
    s = p.get("scales")
    if s is None:
        s = p["scale_codes"].float() / 127 * p["absmax"].repeat_interleave(256)[
            :p["scale_codes"].numel()]
    return (lv[c.int()] * s[:, None]).view(p["rows"], p["cols"]).double()


def _adapter(g, out, inp, r):
    a = (torch.rand(r, inp, device=DEV, generator=g) * 2 - 1) / math.sqrt(inp)
    return a, _randn(g, out, r, std=0.01)


def _dtype(case):
    return torch.bfloat16 if case["act"] == "bf16" else torch.float32


ALPHA = 16.0


def _layer_inputs(case, seed):
    g = _gen(seed)
    n, k, m, t = case["out"], case["inp"], case["tokens"], _dtype(case)
    p = _packed(g, n, k, case["dq"])
    a, b = _adapter(g, n, k, case["r"])
    x = _randn(g, m, k).to(t)
    dy = _randn(g, m, n).to(t) if case["train"] else None
    return p, a, b, x, dy


def _decode_inputs(case, seed):
    g = _gen(seed)
    layers = []
    for _ in range(case["pairs"]):
        for n, k in ((case["out"], case["inp"]), (case["inp"], case["out"])):
            a, b = _adapter(g, n, k, case["r"])
            layers.append((_packed(g, n, k, case["dq"]), a, b,
                           _randn(g, case["batch"], k).to(_dtype(case))))
    return layers


def _block_inputs(case, seed):
    g = _gen(seed)
    h, kv, it, s, r = (case[k] for k in ("hidden", "kv", "inter", "seq", "r"))
    shapes = dict(q=(h, h), k=(kv, h), v=(kv, h), o=(h, h), gate=(it, h), up=(it, h),
                  down=(h, it))
    d = dict(w={n: _packed(g, *sh, True) for n, sh in shapes.items()},
             ab={n: _adapter(g, *sh, r) for n, sh in shapes.items()},
             attn_norm=1 + _randn(g, h, std=0.1), mlp_norm=1 + _randn(g, h, std=0.1),
             x=_randn(g, s, h), attn=_randn(g, s, h))
    if case["train"]:
        d.update(dx=_randn(g, s, h), dq=_randn(g, s, h), dk=_randn(g, s, kv),
                 dv=_randn(g, s, kv))
    return d


def _adam_inputs(case, seed):
    """Per tensor: parameter, an earlier step's gradient, this step's."""
    g = _gen(seed)
    out = []
    for _ in range(case["layers"]):
        for n, k in ((case["out"], case["inp"]), (case["inp"], case["out"])):
            for size in (case["r"] * k, n * case["r"]):
                out.append((_randn(g, size, std=0.02), _randn(g, size, std=0.01),
                            _randn(g, size, std=0.01)))
    return out


def _loss_inputs(case, seed):
    g = _gen(seed)
    logits = _randn(g, case["seq"], case["vocab"], std=3.0)
    return logits, torch.randint(0, case["vocab"], (case["seq"],), device=DEV,
                                 dtype=torch.int32, generator=g)


# ---- what a user's program has in hand ---------------------------------------
def prepare(case, seed):
    kind = case["kind"]
    if kind == "layer":
        p, a, b, x, dy = _layer_inputs(case, seed)
        m, n, k, r = case["tokens"], case["out"], case["inp"], case["r"]
        e = lambda *s: torch.empty(*s, device=DEV)  # noqa: E731
        st = dict(kind=kind, w=_weight(p), lora=QD.lora_struct(a, b, r, ALPHA), x=x, dy=dy,
                  m=m, y=e(m, n), t1=e(m, r))
        st["qw"] = st["w"].struct()
        if dy is not None:
            st.update(gx=e(m, k), ga=e(r, k), gb=e(n, r))
        return st
    if kind == "decode":
        layers, m = [], case["batch"]
        for p, a, b, x in _decode_inputs(case, seed):
            w = _weight(p)
            layers.append((w, QD.lora_struct(a, b, case["r"], ALPHA), x,
                           torch.empty(m, w.rows, device=DEV), None))

        def step():
            for i in range(0, len(layers), 2):
                QD.forward_group(layers[i:i + 2], m)
        step()
        torch.cuda.synchronize()
        graph = torch.cuda.CUDAGraph()
        with torch.cuda.graph(graph):
            step()
        return dict(kind=kind, graph=graph, layers=layers, ys=[L[3] for L in layers])
    if kind == "block":
        d = _block_inputs(case, seed)
        w = {n: _weight(p) for n, p in d["w"].items()}
        lo = {n: (a, b, case["r"], ALPHA) for n, (a, b) in d["ab"].items()}
        at = QD.AttnProjections(d["attn_norm"], *(w[n] for n in "qkvo"),
                                loras=[lo[n] for n in "qkvo"], eps=EPS)
        ml = QD.MLPBlock(d["mlp_norm"], *(w[n] for n in ("gate", "up", "down")),
                         loras=[lo[n] for n in ("gate", "up", "down")], eps=EPS)
        ac, mc = at.new_cache(case["seq"], DEV), ml.new_cache(case["seq"], DEV)
        ac["attn"].copy_(d["attn"])  # the attention's output is the caller's
        return dict(kind=kind, at=at, ml=ml, ac=ac, mc=mc, refs=(w, lo),
                    **{n: d.get(n) for n in ("x", "dx", "dq", "dk", "dv")})
    if kind == "quantize":
        g = _gen(seed)
        return dict(kind=kind, w=_randn(g, case["out"], case["inp"], std=0.02), dq=case["dq"])
    if kind == "adam":
        ts = _adam_inputs(case, seed)
        opt = QH.Adam8bit(lr=1e-3, max_resident_pages=case["pages"] or None)
        n = len(ts)
        arr = lambda i: (C.c_void_p * n)(*[t[i].data_ptr() for t in ts])  # noqa: E731
        st = dict(kind=kind, opt=opt, ts=ts, n=n, p=arr(0), g=arr(2),
                  lens=(C.c_size_t * n)(*[t[0].numel() for t in ts]), stats=QH._lib.AdamStats())
        _adam_step(st, arr(1))  # the optimizer has state from an earlier step
        return st
    logits, targets = _loss_inputs(case, seed)
    return dict(kind=kind, logits=logits, targets=targets, d=torch.empty_like(logits))


def _adam_step(st, grads):
    ctx = st["opt"].ctx
    QH._lib.check(ctx.lib.qh_adam8bit_step_dev(
        st["opt"].h, st["p"], grads, st["lens"], st["n"], C.byref(st["stats"]),
        C.c_void_p(torch.cuda.current_stream().cuda_stream)))


# ---- one pass ------------------------------------------------------------------
def run(st):
    kind = st["kind"]
    if kind == "layer":
        QD.forward(st["w"], st["lora"], st["x"], st["m"], st["y"], t1=st["t1"], qw=st["qw"])
        if st["dy"] is None:
            return [st["y"], st["t1"]]
        QD.backward(st["w"], st["lora"], st["x"], st["dy"], st["m"], st["gx"], st["ga"],
                    st["gb"], t1=st["t1"], qw=st["qw"])
        return [st["y"], st["t1"], st["gx"], st["ga"], st["gb"]]
    if kind == "decode":
        st["graph"].replay()
        return st["ys"]
    if kind == "block":
        at, ml, ac, mc = st["at"], st["ml"], st["ac"], st["mc"]
        x = st["x"].clone()  # the residual stream is updated in place
        q, k, v = at.qkv_forward(x, ac)
        at.o_forward(x, ac)
        ml.forward(x, mc)
        out = [q, k, v, x]
        if st["dx"] is not None:
            dmid, gm = ml.backward(mc, st["dx"])
            dattn, go = at.o_backward(ac, dmid)
            dx, ga = at.qkv_backward(ac, st["dq"], st["dk"], st["dv"], dmid)
            out += [dmid, dattn, dx]
            for a, b in [*gm, go, *ga]:
                out += [a, b]
        return out
    if kind == "quantize":
        q = QD.DeviceWeight.quantize(st["w"], 64, st["dq"])
        return [q.codes, q.scale_codes, q.absmax] if st["dq"] else [q.codes, q.scales]
    if kind == "adam":
        _adam_step(st, st["g"])
        return [t[0] for t in st["ts"]]
    return list(QD.softmax_cross_entropy(st["logits"], st["targets"], dlogits=st["d"]))


# ---- the work of one pass -------------------------------------------------------
def _wbytes(n, k, dq):
    e = n * k
    return e / 2 + (e / 64 + 4 * math.ceil(e / 16384) if dq else e / 16)


def _layer_work(n, k, m, r, es, dq, train):
    """(bytes, flops) of one projection: weight, adapter, x and y, and in
    training dy, the input gradient and the adapter's gradients."""
    by = _wbytes(n, k, dq) + 4 * r * (n + k) + es * m * k + 4 * m * n
    fl = 2 * m * n * k + 2 * m * r * (n + k)
    if train:
        by += es * m * n + 4 * m * k + 4 * r * (n + k)
        fl += 2 * m * n * k + 4 * m * r * (n + k)
    return by, fl


def work(case):
    kind = case["kind"]
    if kind in ("layer", "decode"):
        es = 2 if case["act"] == "bf16" else 4
        n, k, r = case["out"], case["inp"], case["r"]
        if kind == "layer":
            by, fl = _layer_work(n, k, case["tokens"], r, es, case["dq"], case["train"])
        else:
            ws = [_layer_work(*s, case["batch"], r, es, case["dq"], False)
                  for s in ((n, k), (k, n))]
            by, fl = (case["pairs"] * sum(w[i] for w in ws) for i in (0, 1))
        return dict(bytes=by, flops=fl)
    if kind == "block":
        h, kv, it, s, r, tr = (case[k] for k in ("hidden", "kv", "inter", "seq", "r", "train"))
        by = fl = 0
        for n, k in ((h, h), (kv, h), (kv, h), (h, h), (it, h), (it, h), (h, it)):
            b, f = _layer_work(n, k, s, r, 4, True, tr)
            by, fl = by + b, fl + f
        return dict(bytes=by, flops=fl)
    if kind == "quantize":
        n, k = case["out"], case["inp"]
        return dict(bytes=4 * n * k + _wbytes(n, k, case["dq"]), flops=0)
    if kind == "adam":
        e = case["layers"] * 2 * case["r"] * (case["out"] + case["inp"])
        return dict(bytes=16 * e + 16 * e / 256, flops=0)
    return dict(bytes=8 * case["seq"] * case["vocab"], flops=0)


# ---- how far another correct implementation may be off --------------------------
def tolerance(case):
    kind = case["kind"]
    if kind in ("quantize", "adam"):
        return "exact"  # the reference's bits
    if kind == "loss":
        return dict(rel=1e-6)  # fp32 exponentials and sums: 4e-8 measured
    # about four times the error against 64 bits: products of fp32 values in
    # split bf16 parts, 2.5e-6 to 6.3e-6 in one layer, 1.1e-5 through a block
    return dict(rel=4e-5 if kind == "block" else 2e-5)


# ---- the same in 64 bits ----------------------------------------------------------
def _proj(p, ab, r, x):
    a, b = (t.double() for t in ab)
    w = _dense(p)
    t1 = x @ a.T
    return x @ w.T + (ALPHA / r) * (t1 @ b.T), t1


def _proj_back(p, ab, r, x, dy):
    a, b = (t.double() for t in ab)
    ds = (ALPHA / r) * (dy @ b)
    return dy @ _dense(p) + ds @ a, ds.T @ x, (ALPHA / r) * (dy.T @ (x @ a.T))


def _norm(x, w):
    return x / torch.sqrt((x * x).mean(1, keepdim=True) + EPS) * w


def _norm_back(x, w, dy):
    rs = 1 / torch.sqrt((x * x).mean(1, keepdim=True) + EPS)
    t = dy * w
    return rs * t - x * rs ** 3 * (t * x).mean(1, keepdim=True)


def exact(case, seed):
    kind = case["kind"]
    if kind == "layer":
        p, a, b, x, dy = _layer_inputs(case, seed)
        y, t1 = _proj(p, (a, b), case["r"], x.double())
        if dy is None:
            return [y, t1]
        gx, ga, gb = _proj_back(p, (a, b), case["r"], x.double(), dy.double())
        return [y, t1, gx, ga, gb]
    if kind == "decode":
        return [_proj(p, (a, b), case["r"], x.double())[0]
                for p, a, b, x in _decode_inputs(case, seed)]
    if kind == "block":
        return _block_exact(case, _block_inputs(case, seed))
    if kind == "quantize":
        w = _randn(_gen(seed), case["out"], case["inp"], std=0.02).view(-1, 64)
        s = w.abs().amax(1)
        if not case["dq"]:
            return [None, s]
        nb = s.numel()
        return [None, None, torch.nn.functional.pad(s, (0, -nb % 256)).view(-1, 256).amax(1)]
    if kind == "adam":
        return [_adam_exact(*(t.double() for t in ts)) for ts in _adam_inputs(case, seed)]
    logits, targets = _loss_inputs(case, seed)
    lp = torch.log_softmax(logits.double(), 1)
    del logits
    rows = torch.arange(case["seq"], device=DEV)
    loss = -lp[rows, targets.long()].mean().view(1)
    d = lp.exp_()
    d[rows, targets.long()] -= 1
    return [loss, d / case["seq"]]


def _block_exact(case, d):
    r = case["r"]
    f = lambda n, x: _proj(d["w"][n], d["ab"][n], r, x)[0]  # noqa: E731
    bk = lambda n, x, dy: _proj_back(d["w"][n], d["ab"][n], r, x, dy)  # noqa: E731
    x, attn = d["x"].double(), d["attn"].double()
    an, mn = d["attn_norm"].double(), d["mlp_norm"].double()
    xa = _norm(x, an)
    q, k, v = (f(n, xa) for n in "qkv")
    mid = x + f("o", attn)
    xm = _norm(mid, mn)
    gate, up = f("gate", xm), f("up", xm)
    act = torch.nn.functional.silu(gate) * up
    out = [q, k, v, mid + f("down", act)]
    if not case["train"]:
        return out
    dx, dq, dk, dv = (d[n].double() for n in ("dx", "dq", "dk", "dv"))
    dact, da, db = bk("down", act, dx)
    g_down = [da, db]
    sg = torch.sigmoid(gate)
    dgate = dact * up * sg * (1 + gate * (1 - sg))
    dup = dact * gate * sg
    d1, *g_gate = bk("gate", xm, dgate)
    d2, *g_up = bk("up", xm, dup)
    dmid = dx + _norm_back(mid, mn, d1 + d2)
    dattn, *g_o = bk("o", attn, dmid)
    s, grads = 0, []
    for n, t in (("q", dq), ("k", dk), ("v", dv)):
        t, *gr = bk(n, xa, t)
        s, grads = s + t, grads + gr
    out += [dmid, dattn, dmid + _norm_back(x, an, s)]
    grads = g_gate + g_up + g_down + g_o + grads
    return out + [t.reshape(-1) for t in grads]


def _adam_exact(p, g1, g2):
    """Two steps of Adam whose moments (the second as its root) go through
    int8 codes per 256 elements after the first."""
    def q8(t):
        n = t.numel()
        b = torch.nn.functional.pad(t, (0, -n % 256)).view(-1, 256)
        s = b.abs().amax(1, keepdim=True)
        x = b / s * 127
        c = torch.trunc(x + torch.sign(x) * 0.5)
        return (c / 127 * s).view(-1)[:n]
    # the configuration's fp32 values
    b1, b2, lr, eps = (float(torch.tensor(v)) for v in (0.9, 0.999, 1e-3, 1e-8))
    m = v = torch.zeros_like(p)
    for t, g in ((1, g1), (2, g2)):
        m = b1 * m + (1 - b1) * g
        var = b2 * v * v + (1 - b2) * g * g
        p = p - lr * (m / (1 - b1 ** t)) / (torch.sqrt(var / (1 - b2 ** t)) + eps)
        m, v = q8(m), q8(torch.sqrt(var))
    return p
