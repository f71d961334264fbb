"""Head dim 256 in fp16/bf16 at the edges of its tiles (64 queries or keys per
workgroup, 16 per wave, 32-key and 32-query tiles): one token, remainders of
every tile, window and prefix edges inside a tile, grouped heads, a strided
layout and padded head dims, each forward and backward in full against the
fp64 oracle (tolerances of ``tests/parity_util.py``)."""
import pytest
import torch

from cron_root_attention.core import _attention_with_plan
from oracle import cra_oracle as O
from tests.parity_util import BF16, DEV, F16, TOL_GRAD, check_forward, inputs, rel_fro, say

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("S,W,relay,D,Hq,Hkv,dtype,bshd", [
    (1, 1, False, 256, 1, 1, F16, False),
    (15, 4, False, 256, 2, 1, BF16, False),
    (33, 6, False, 256, 1, 1, F16, True),
    (64, 8, True, 256, 2, 2, F16, False),
    (65, 32, True, 256, 2, 1, BF16, True),   # a window of one key tile
    (97, 33, True, 200, 1, 1, F16, False),   # padded head dim, a tile and one key
    (257, 17, True, 256, 4, 1, BF16, True),
    (640, 5, True, 129, 2, 2, F16, False),   # 384 global rows
])
def test_edges(S, W, relay, D, Hq, Hkv, dtype, bshd):
    say(f"wide tiles: S={S} W={W} relay={relay} D={D} H={Hq}/{Hkv} {dtype} bshd={bshd}")
    q, k, v, do = inputs(1, Hq, Hkv, S, D, dtype, seed=S)
    plan = O.Plan(S, W, relay, 2)

    def dev(t):
        t = t.to(DEV)
        return t.transpose(1, 2).contiguous().transpose(1, 2) if bshd else t

    x = [dev(t).requires_grad_(True) for t in (q, k, v)]
    o = _attention_with_plan(*x, W, relay, Hq // Hkv)
    check_forward(o, q, k, v, plan, dtype, kv_groups=Hq // Hkv)
    _, _, _, ref = O.forward_backward(q, k, v, do, plan, kv_groups=Hq // Hkv)
    got = torch.autograd.grad(o, x, dev(do))
    for name, t in zip(("dq", "dk", "dv"), got):
        # one key: its softmax is constant, dq and dk are zero up to rounding
        if S == 1 and name != "dv":
            assert float(t.abs().max()) <= 2 * TOL_GRAD[dtype]
            continue
        e = rel_fro(t, ref[name])
        say(f"  {name}: rel {e:.3e}")
        assert e <= TOL_GRAD[dtype], name
