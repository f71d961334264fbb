"""Performance cases of the sqrt(N) sparse attention on one GPU.

Every case is one pass of work that a program built on this package has it do,
through the public entry points: ``cron_root_attention`` (forward under
no_grad, or a training step with the gradients of q, k, v), its packed form
``cron_root_attention_varlen`` and the layer ``CronRootAttention``.  A case is
a dict of plain values:

    api     "attention", "varlen" or "layer"
    train   forward + backward (True) or forward alone
    B, Hq, Hkv, S, D, dtype      problem sizes; Hkv < Hq is grouped-query attention
    bshd    q, k, v are [B, S, H, D] buffers viewed as [B, H, S, D], as a
            projection leaves them (otherwise contiguous [B, H, S, D])
    scale   a relay_log_scale parameter is passed (and gets its gradient)
    top_k   relay rows per block
    docs    varlen only: document lengths, comma separated
"""
import math
import os
import sys

import torch

_PKG = os.path.join(os.path.dirname(os.path.dirname(os.path.abspath(__file__))), "cron-root-attention_amd")
if _PKG not in sys.path:
    sys.path.insert(0, _PKG)

import cron_root_attention as cra  # noqa: E402

_DTYPES = {"f16": torch.float16, "bf16": torch.bfloat16, "f32": torch.float32}


def _case(name, api, train, B, Hq, Hkv, S, D, dtype, bshd=False, scale=False, top_k=2, docs=""):
    c = dict(api=api, train=train, B=B, Hq=Hq, Hkv=Hkv, S=S, D=D, dtype=dtype, bshd=bshd, scale=scale,
             top_k=top_k, docs=docs)
    return dict(c, name=name) if name else c


# Document lengths of one packed training batch: a few long documents, many
# short ones, odd lengths, one of a single token.
_DOCS = (9001, 4096, 3333, 2049, 2048, 1500, 1023, 1000, 640, 511, 300, 257, 129, 64, 17, 1)


def listed():
    return [
        # a short prompt through a small model: a call of launches and host time
        _case("fwd_512", "attention", False, 1, 8, 8, 512, 64, "f16"),
        # a training step on one short, odd-length sequence of a small model
        _case("train_1k", "attention", True, 1, 12, 12, 1000, 64, "bf16", bshd=True),
        # prefill of a medium prompt through a small model, relay rows on
        _case("fwd_8k", "attention", False, 1, 8, 8, 8192, 64, "f16"),
        # training an XL model at an ordinary context length, two sequences a GPU
        _case("train_4k", "attention", True, 2, 32, 32, 4096, 128, "bf16"),
        # long-context training of a medium model
        _case("train_32k", "attention", True, 1, 12, 12, 32768, 64, "f16"),
        # the benchmark shape: prefill and training at 128K tokens
        _case("fwd_128k", "attention", False, 1, 16, 16, 131072, 128, "f16"),
        _case("train_128k", "attention", True, 1, 16, 16, 131072, 128, "f16"),
        # the longest context in use
        _case("fwd_512k", "attention", False, 1, 16, 16, 524288, 128, "f16"),
        # one packed batch of documents, grouped kv heads, projection layout
        _case("varlen_26k", "varlen", True, 1, 16, 4, sum(_DOCS), 128, "bf16", bshd=True,
              docs=",".join(str(n) for n in _DOCS)),
        # full-precision training at the size the fp32 reference is quoted on
        _case("train_f32_4k", "attention", True, 1, 8, 8, 4096, 64, "f32"),
        # wide heads, grouped, an odd length, a learned relay scale
        _case("train_wide_8k", "attention", True, 1, 8, 4, 8191, 256, "bf16", scale=True),
        # the whole layer: projections, attention, output projection, all gradients
        _case("layer_16k", "layer", True, 1, 16, 4, 16000, 128, "bf16"),
    ]


# ---------------------------------------------------------------------------
# sizes
# ---------------------------------------------------------------------------
def _lens(case):
    return [int(x) for x in case["docs"].split(",")] if case["docs"] else [case["S"]]


def _window(n):
    return int(math.ceil(math.sqrt(n)))  # the op's rule


def _pairs(n, top_k):
    """(query, key) pairs of one head of a sequence of n tokens."""
    W = _window(n)
    i = torch.arange(n, dtype=torch.int64)
    ls = (i - W + 1).clamp_min(0)
    rel = top_k * (ls // W) if n > 2048 else torch.zeros_like(ls)  # relay rows above 2048 tokens
    return int(((i + 1).clamp_max(W) + (ls + W - 1) // W + rel).sum())


def work(case):
    B, Hq, Hkv, S, D = (case[x] for x in ("B", "Hq", "Hkv", "S", "D"))
    e = 4 if case["dtype"] == "f32" else 2
    pairs = sum(_pairs(n, case["top_k"]) for n in _lens(case)) * B * Hq
    q, kv = B * Hq * S * D * e, B * Hkv * S * D * e
    # scores and P.V; a backward adds five products (S again, dP, dQ, dK, dV)
    flops = (14 if case["train"] else 4) * D * pairs
    if case["api"] != "layer":
        # q, k, v in, o out; a step also dO in, dq, dk, dv out
        return {"bytes": (4 * q + 4 * kv) if case["train"] else (2 * q + 2 * kv), "flops": flops}
    dm = Hq * D
    mats = dm * (2 * dm + 2 * Hkv * D)  # q, o, k and v projection weights
    x = B * S * dm * e
    # x and weights in, y out; a step also dy in, dx and the weights' gradients out
    return {"bytes": (4 if case["train"] else 2) * x + (2 if case["train"] else 1) * mats * e,
            "flops": flops + (6 if case["train"] else 2) * B * S * mats}


def _cost(case):
    """Bound on a case's share of the GPU: its products, weighted by how fast the
    matrix cores take its type, and the memory it holds."""
    w = work(case)
    slow = 30 if case["dtype"] == "f32" else 9 if case["D"] > 128 else 2.5 if case["train"] else 1.5
    return w["flops"] * slow, w["bytes"]


_LARGEST = None


def _fits(case):
    global _LARGEST
    if _LARGEST is None:
        _LARGEST = _cost(next(c for c in listed() if c["name"] == "fwd_512k"))
    c = _cost(case)
    return c[0] <= _LARGEST[0] and c[1] <= _LARGEST[1]


def _log_int(rng, lo, hi):
    return int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))


def draw(rng):
    api = rng.choice(["attention"] * 6 + ["varlen"] * 2 + ["layer"])
    train = rng.random() < 0.6
    D = rng.choice([32, 64, 64, 64, 80, 96, 128, 128, 128, 128, 256])
    dtype = rng.choice(["f16", "f16", "f16", "bf16", "bf16", "bf16", "f32"])
    if api == "layer":
        D, dtype = rng.choice([64, 128]), "bf16"
    grp = rng.choice([1, 1, 1, 2, 4, 8])
    Hkv = rng.choice([1, 2, 3, 4, 6, 8, 12, 16, 32])
    while grp * Hkv > 64:
        grp //= 2
    Hq = grp * Hkv
    if api == "layer":  # a model width
        Hkv, grp = rng.choice([(4, 4), (8, 1), (8, 2), (8, 4), (12, 1), (16, 1)])
        Hq = Hkv * grp
    B = rng.choice([1, 1, 1, 2, 3, 4])
    bshd = rng.random() < 0.5
    scale = api != "layer" and rng.random() < 0.2
    top_k = rng.choice([2, 2, 2, 1, 4]) if api == "attention" else 2
    if api == "varlen":
        B = 1
        lens = [_log_int(rng, 1, 16384) for _ in range(_log_int(rng, 2, 48))]
        while True:
            c = _case(None, api, train, B, Hq, Hkv, sum(lens), D, dtype, bshd, scale, top_k,
                      ",".join(str(n) for n in lens))
            if _fits(c) or len(lens) == 2:
                return c
            lens.pop()
    S = _log_int(rng, 16, 524288)
    while True:
        c = _case(None, api, train, B, Hq, Hkv, S, D, dtype, bshd, scale, top_k)
        if _fits(c):
            return c
        S = max(16, int(S * 0.6))


# ---------------------------------------------------------------------------
# inputs and the pass
# ---------------------------------------------------------------------------
def _inputs(case, seed):
    dev = torch.device("cuda")
    gen = torch.Generator(device=dev).manual_seed(seed)
    dt = _DTYPES[case["dtype"]]
    B, Hq, Hkv, S, D = (case[x] for x in ("B", "Hq", "Hkv", "S", "D"))

    def normal(*shape):
        return torch.randn(*shape, generator=gen, device=dev, dtype=torch.float32).to(dt)

    def heads(H):
        if case["bshd"]:
            return normal(B, S, H, D).transpose(1, 2)
        return normal(B, H, S, D)

    if case["api"] == "layer":
        dm = Hq * D
        mods = {n: normal(o, dm) * math.sqrt(2.0 / (o + dm))
                for n, o in (("q", dm), ("k", Hkv * D), ("v", Hkv * D), ("o", dm))}
        return {"x": normal(B, S, dm), "w": mods, "dy": normal(B, S, dm)}
    t = {"q": heads(Hq), "k": heads(Hkv), "v": heads(Hkv), "do": heads(Hq) if case["train"] else None}
    t["alpha"] = (0.3 * torch.randn(Hkv, generator=gen, device=dev)) if case["scale"] else None
    return t


def prepare(case, seed):
    t = _inputs(case, seed)
    if case["api"] == "layer":
        layer = cra.CronRootAttention(case["Hq"] * case["D"], case["Hq"], n_kv_heads=case["Hkv"], hybrid=True)
        layer = layer.to(device="cuda", dtype=_DTYPES[case["dtype"]]).train(case["train"])
        with torch.no_grad():
            for n, w in t["w"].items():
                getattr(layer, n + "_proj").weight.copy_(w)
        leaves = [t["x"], *(getattr(layer, n + "_proj").weight for n in "qkvo")]
        t["x"].requires_grad_(case["train"])
        return {"api": "layer", "train": case["train"], "layer": layer, "x": t["x"], "dy": t["dy"], "leaves": leaves}
    args = dict(kv_groups=case["Hq"] // case["Hkv"], relay_top_k=case["top_k"])
    leaves = [t["q"], t["k"], t["v"]] + ([t["alpha"]] if case["scale"] else [])
    if case["train"]:
        for x in leaves:
            x.requires_grad_(True)
    if case["scale"]:
        args["relay_log_scale"] = t["alpha"]
    if case["api"] == "varlen":
        cu = [0]
        for n in _lens(case):
            cu.append(cu[-1] + n)
        args["cu_seqlens"] = cu
    # without a relay row (at most 2048 tokens) the scale is unused and has no gradient
    if case["scale"] and max(_lens(case)) <= 2048:
        leaves = leaves[:3]
    return {"api": case["api"], "train": case["train"], "qkv": (t["q"], t["k"], t["v"]), "do": t["do"],
            "args": args, "leaves": leaves}


def run(state):
    if state["api"] == "layer":
        if not state["train"]:
            with torch.no_grad():
                return state["layer"](state["x"])
        y = state["layer"](state["x"])
        return [y.detach(), *torch.autograd.grad(y, state["leaves"], state["dy"])]
    op = cra.cron_root_attention_varlen if state["api"] == "varlen" else cra.cron_root_attention
    if not state["train"]:
        with torch.no_grad():
            return op(*state["qkv"], **state["args"])
    o = op(*state["qkv"], **state["args"])
    return [o.detach(), *torch.autograd.grad(o, state["leaves"], state["do"])]


# ---------------------------------------------------------------------------
# the same in 64 bits, in plain torch
# ---------------------------------------------------------------------------
def _bmm(a, b):
    return torch.bmm(a, b.contiguous())


def _exact_sequence(q, k, v, do, top_k, alpha):
    """One sequence of [B, H, n, D] tensors; returns o and, with do, dq, dk,
    dv and d(alpha) ([H_kv], when alpha is given). A query sees its window of
    W = ceil(sqrt(n)) tokens and a prefix of the global rows: of every earlier
    W-block its first row, then (n > 2048) its top_k rows of largest norm."""
    B, Hq, n, D = q.shape
    Hkv = k.shape[1]
    grp = Hq // Hkv
    dev = q.device
    W = _window(n)
    nb, full = (n + W - 1) // W, n // W
    relay = n > 2048
    rpb = 1 + top_k if relay else 1
    BH = B * Hkv
    rows = torch.zeros(BH, nb, rpb, dtype=torch.int64, device=dev)  # source row of each global row
    rows[:, :, 0] = torch.arange(nb, device=dev) * W
    mul = torch.ones(BH, nb, rpb, dtype=torch.float64, device=dev)
    k2, v2 = k.reshape(BH, n, D), v.reshape(BH, n, D)
    if relay:
        norm = torch.stack([k2[i].double().square().sum(-1) for i in range(BH)])[:, :full * W]
        best = norm.view(BH, full, W).sort(dim=-1, descending=True, stable=True).indices[..., :top_k]
        rows[:, :full, 1:] = best + (torch.arange(full, device=dev) * W)[None, :, None]
        if full < nb:  # no query sees the relay rows of a partial block
            rows[:, full:, 1:] = full * W
        if alpha is not None:
            mul[:, :, 1:] = alpha.double().exp().repeat(B)[:, None, None]
    rows, mul = rows.view(BH, -1), mul.view(BH, -1, 1)
    idx = rows[:, :, None].expand(-1, -1, D)
    gk, gv = k2.gather(1, idx).double() * mul, v2.gather(1, idx).double() * mul
    o = torch.empty(BH, grp, n, D, dtype=torch.float64, device=dev)
    train = do is not None
    if train:
        dq = torch.empty_like(o)
        dk, dv = (torch.zeros(BH, n, D, dtype=torch.float64, device=dev) for _ in range(2))
        dgk, dgv = torch.zeros_like(gk), torch.zeros_like(gv)
        do2 = do.reshape(BH, grp, n, D)
    q2 = q.reshape(BH, grp, n, D)
    C = max(128, min(1024, W))  # queries per step
    for m0 in range(0, n, C):
        m1 = min(n, m0 + C)
        lo = max(0, m0 - W + 1)
        i = torch.arange(m0, m1, device=dev)
        ls = (i - W + 1).clamp_min(0)
        pre = rpb * (ls // W) + (ls % W != 0).long()
        G = int(pre[-1])
        j = torch.arange(lo, m1, device=dev)
        see = torch.cat([(j[None] <= i[:, None]) & (j[None] >= ls[:, None]),
                         torch.arange(G, device=dev)[None] < pre[:, None]], 1)
        kk = torch.cat([k2[:, lo:m1].double(), gk[:, :G]], 1)
        vv = torch.cat([v2[:, lo:m1].double(), gv[:, :G]], 1)
        for g in range(grp):
            qc = q2[:, g, m0:m1].double()
            s = _bmm(qc, kk.transpose(1, 2)) / math.sqrt(D)
            p = s.masked_fill_(~see[None], -math.inf).softmax(-1)
            oc = _bmm(p, vv)
            o[:, g, m0:m1] = oc
            if not train:
                continue
            dc = do2[:, g, m0:m1].double()
            ds = _bmm(dc, vv.transpose(1, 2))
            ds = (ds - (oc * dc).sum(-1, keepdim=True)) * p / math.sqrt(D)
            dq[:, g, m0:m1] = _bmm(ds, kk)
            dkk = torch.bmm(ds.transpose(1, 2).contiguous(), qc)
            dvv = torch.bmm(p.transpose(1, 2).contiguous(), dc)
            n_loc = m1 - lo
            dk[:, lo:m1] += dkk[:, :n_loc]
            dv[:, lo:m1] += dvv[:, :n_loc]
            dgk[:, :G] += dkk[:, n_loc:]
            dgv[:, :G] += dvv[:, n_loc:]
    if not train:
        return (o.view(B, Hq, n, D),)
    dk.scatter_add_(1, idx, dgk * mul)
    dv.scatter_add_(1, idx, dgv * mul)
    da = None
    if alpha is not None:
        da = torch.zeros(BH, dtype=torch.float64, device=dev)
        if relay:
            both = (dgk * gk + dgv * gv).sum(-1).view(BH, nb, rpb)
            da = both[:, :, 1:].sum((1, 2))
        da = da.view(B, Hkv).sum(0)
    return o.view(B, Hq, n, D), dq.view(B, Hq, n, D), dk.view(B, Hkv, n, D), dv.view(B, Hkv, n, D), da


def _exact_attention(case, q, k, v, do, alpha):
    outs, at = [], 0
    for n in _lens(case):
        c = [x if x is None else x[:, :, at:at + n] for x in (q, k, v, do)]
        outs.append(_exact_sequence(*c, case["top_k"], alpha))
        at += n
    r = [torch.cat(x, 2) for x in list(zip(*outs))[:4]]
    if do is not None and alpha is not None:
        r.append(sum(x[4] for x in outs))
    return r


def exact(case, seed):
    t = _inputs(case, seed)
    with torch.no_grad():
        if case["api"] != "layer":
            r = _exact_attention(case, t["q"], t["k"], t["v"], t["do"], t["alpha"])
            if not case["train"]:
                return r[0]
            return r[:4] if max(_lens(case)) <= 2048 else r
        B, S, D = case["B"], case["S"], case["D"]
        x = t["x"].double()
        w = {n: m.double() for n, m in t["w"].items()}

        def split(y):
            return y.view(B, S, -1, D).transpose(1, 2)

        def join(y):
            return y.transpose(1, 2).reshape(B, S, -1)

        # the projections' results are in the layer's type: the relay rows are chosen among those
        q, k, v = (split((x @ w[n].t()).to(t["x"].dtype)) for n in "qkv")
        if not case["train"]:
            o = join(_exact_attention(case, q, k, v, None, None)[0])
            return o @ w["o"].t()
        dy = t["dy"].double()
        do = dy @ w["o"]
        o, dq, dk, dv = _exact_attention(case, q, k, v, split(do), None)
        o, dq, dk, dv = (join(y) for y in (o, dq, dk, dv))
        two = [y.reshape(B * S, -1) for y in (x, dy, o, dq, dk, dv)]
        dx = dq @ w["q"] + dk @ w["k"] + dv @ w["v"]
        return [o @ w["o"].t(), dx, two[3].t() @ two[0], two[4].t() @ two[0], two[5].t() @ two[0],
                two[1].t() @ two[2]]


def tolerance(case):
    # About four times the distance from exact() (2-norm, the largest of a
    # case's outputs) measured over the listed cases and drawn ones: f16 2.8e-4
    # forward and 3.0e-4 gradients (2.9e-4 at 512K tokens), bf16 2.5e-3, f32
    # 3.4e-7 to 1.5e-6; with a relay scale 1.2e-3 and (d(alpha)) 1.7e-2, where
    # exp(alpha) and the scaled rows are rounded to the input type; the layer 4e-3.
    if case["api"] == "layer":
        return {"rel": 1.6e-2}
    if case["scale"]:
        return {"rel": {"f16": 5e-3, "bf16": 3e-2, "f32": 6e-6}[case["dtype"]]}
    return {"rel": {"f16": 1.2e-3, "bf16": 1e-2, "f32": 6e-6}[case["dtype"]]}
