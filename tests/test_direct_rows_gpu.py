"""Sequences without relay, whose global rows the kernels read in k and v:
against the same launch over packed rows (the phase-restricted and persistent
forms always read those) and the fp64 oracle, at tile edges, in strided and
GQA layouts, every type and head dim."""
import pytest
import torch

import cron_root_attention as cra
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
