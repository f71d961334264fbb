"""Sequences without relay, whose global rows the kernels read in k and v:
against the same call over packed rows (the persistent form's, and where k and
v have different strides) and the fp64 oracle, at tile edges, in strided and
GQA layouts, every type and head dim; and packed rows of a caller's own."""
import math

import pytest
import torch

import cron_root_attention as cra
from cron_root_attention import _native
from cron_root_attention.core import CronRootAttentionV14Function
from oracle import cra_oracle as O
from tests.parity_util import BF16, DEV, F16, F32, TOL_GRAD, check_forward, inputs, rel_fro, say

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("B,Hq,Hkv,S,D,dtype,bshd", [
    (1, 1, 1, 1, 64, F16, False),
    (2, 4, 2, 129, 64, F16, True),
    (1, 2, 2, 2048, 64, BF16, False),   # the longest without relay
    (1, 6, 3, 1000, 128, F16, True),
    (1, 3, 1, 511, 128, BF16, False),   # odd head count: XCD-aware order
    (2, 2, 2, 300, 32, F16, True),
    (1, 2, 1, 777, 256, F16, True),
    (1, 2, 2, 400, 96, BF16, False),    # padded head dim
    (2, 2, 1, 650, 64, F32, True),
    (1, 1, 1, 300, 256, F32, False),
])
def test_against_packed_and_oracle(B, Hq, Hkv, S, D, dtype, bshd):
    say(f"direct rows: B={B} H={Hq}/{Hkv} S={S} D={D} {dtype} bshd={bshd}")
    q, k, v, do = inputs(B, Hq, Hkv, S, D, dtype, seed=S + D)

    def dev(t):
        t = t.to(DEV)
        return t.transpose(1, 2).contiguous().transpose(1, 2) if bshd else t

    x = [dev(t).requires_grad_(True) for t in (q, k, v)]
    grp, plan = Hq // Hkv, O.make_plan(S)
    o = cra.cron_root_attention(*x, kv_groups=grp)
    got = torch.autograd.grad(o, x, dev(do))
    op = CronRootAttentionV14Function.apply(*x, True, grp)   # persistent: packed rows
    packed = torch.autograd.grad(op, x, dev(do))
    assert torch.equal(o, op)
    for a, b in zip(got, packed):
        assert torch.equal(a, b)
    check_forward(o, q, k, v, plan, dtype, kv_groups=grp)
    _, _, _, ref = O.forward_backward(q, k, v, do, plan, kv_groups=grp)
    for name, t in zip(("dq", "dk", "dv"), got):
        if S == 1 and name != "dv":  # one key: its softmax is constant
            continue
        assert rel_fro(t, ref[name]) <= TOL_GRAD[dtype], name


@pytest.mark.parametrize("S,D,dtype", [(129, 64, F16), (777, 128, BF16), (400, 256, F16), (300, 64, F32)])
def test_different_strides_are_packed(S, D, dtype):
    """k contiguous, v a projection's [B, S, H, D] buffer: the packed forward and
    backward without relay, against the in-place ones and the fp64 oracle."""
    say(f"packed without relay: S={S} D={D} {dtype}")
    q, k, v, do = inputs(2, 4, 2, S, D, dtype, seed=S)
    x = [t.to(DEV).requires_grad_(True) for t in (q, k, v)]
    y = x[:2] + [x[2].detach().transpose(1, 2).contiguous().transpose(1, 2).requires_grad_(True)]
    p = _native.problem(2, 4, 2, S, D, math.ceil(math.sqrt(S)), False, 2, dtype, 1 / math.sqrt(D))
    assert not _native.reads_global_rows(p, x[1], x[2]) and _native.reads_global_rows(p, y[1], y[2])
    res = []
    for t in (x, y):
        o = cra.cron_root_attention(*t, kv_groups=2)
        res.append([o, *torch.autograd.grad(o, t, do.to(DEV))])
    for a, b in zip(*res):
        assert torch.equal(a, b)
    check_forward(res[1][0], q, k, v, O.make_plan(S), dtype, kv_groups=2)
    _, _, _, ref = O.forward_backward(q, k, v, do, O.make_plan(S), kv_groups=2)
    for name, t in zip(("dq", "dk", "dv"), res[1][1:]):
        assert rel_fro(t, ref[name]) <= TOL_GRAD[dtype], name


@pytest.mark.parametrize("S,D,dtype", [(130, 64, F16), (300, 128, BF16), (200, 256, BF16), (150, 32, F32)])
def test_rows_of_a_callers_own(S, D, dtype):
    """cra_fwd and cra_bwd attend to the packed rows they are given, also where
    they could read the strided rows in k and v."""
    say(f"own global rows: S={S} D={D} {dtype}")
    W = math.ceil(math.sqrt(S))
    G = (S + W - 1) // W
    q, k, v, do = inputs(1, 1, 1, S, D, dtype, seed=S)
    gk, gv, _, _ = inputs(1, 1, 1, G, D, dtype, seed=S + 1)
    p = _native.problem(1, 1, 1, S, D, W, False, 2, dtype, 1 / math.sqrt(D))
    qd, kd, vd, dod, gkd, gvd = (t.to(DEV) for t in (q, k, v, do, gk, gv))
    assert not _native.reads_global_rows(p, kd, vd)
    o, lse = _native.forward(p, qd, kd, vd, gkd, gvd)
    dq, dk, dv, _ = _native.backward(p, qd, kd, vd, o, dod, lse, gkd, gvd, None, None, False)

    leaves = [t[0, 0].double().requires_grad_(True) for t in (q, k, v, gk, gv)]
    q_, k_, v_, gk_, gv_ = leaves
    i, ls = torch.arange(S)[:, None], (torch.arange(S) - W + 1).clamp_min(0)[:, None]
    j, r = torch.arange(S)[None], torch.arange(G)[None]
    see = torch.cat([(j <= i) & (j >= ls), r * W < ls], 1)
    s = (q_ @ torch.cat([k_, gk_]).t() / math.sqrt(D)).masked_fill(~see, -math.inf)
    ref = s.softmax(-1) @ torch.cat([v_, gv_])
    rq, rk, rv, rgk, rgv = torch.autograd.grad(ref, leaves, do[0, 0].double())
    rk[::W] += rgk   # the gradient of a row goes to its strided key
    rv[::W] += rgv
    for name, t, w in (("o", o, ref.detach()), ("dq", dq, rq), ("dk", dk, rk), ("dv", dv, rv)):
        assert rel_fro(t[0, 0], w) <= TOL_GRAD[dtype], name


@pytest.mark.parametrize("D", [64, 80])   # the C++ operator, the Python Function
def test_saved_tensor_hooks_may_change_layouts(D):
    """Nothing is packed in the forward; a hook then gives v back with another
    row stride than k's, for which the kernels would read packed rows."""
    q, k, v, do = (t.to(DEV) for t in inputs(1, 2, 2, 300, D, F16, seed=5))
    x = [t.requires_grad_(True) for t in (q, k, v)]
    want = torch.autograd.grad(cra.cron_root_attention(*x), x, do)
    seen = []

    def unpack(t):
        if t.dim() == 4 and t.shape[2] == 300:
            seen.append(t)
            if len(seen) == 3:  # q, k, v, ...: v as a [B, S, H, D] buffer
                return t.transpose(1, 2).contiguous().transpose(1, 2)
        return t

    with torch.autograd.graph.saved_tensors_hooks(lambda t: t, unpack):
        o = cra.cron_root_attention(*x)
    got = torch.autograd.grad(o, x, do)
    assert len(seen) >= 3
    for a, b in zip(got, want):
        assert torch.equal(a, b)
