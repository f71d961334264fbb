"""fp32 on the bf16 matrix core (every operand cut in three bf16 pieces): tile
edges against the fp64 oracle with the fp32 tolerances, inputs far from 1, and
infinite inputs.

Tolerances: relative Frobenius 2e-6 of o and the gradients. The three left-out
piece products are at most 2^-23 of a product, an fp32 accumulation over n
terms adds about sqrt(n) 2^-24 (n <= 1300 keys or queries here): 1.2e-7 +
36 * 6e-8 = 2.3e-6 at most, and all measured below 6e-7."""
import pytest
import torch

from cron_root_attention.core import _attention_with_plan
from oracle import cra_oracle as O
from tests.parity_util import DEV, F32, inputs, rel_fro, say

pytestmark = pytest.mark.gpu
TOL = 2e-6


def _run(q, k, v, do, W, relay, grp):
    x = [t.to(DEV).requires_grad_(True) for t in (q, k, v)]
    o = _attention_with_plan(*x, W, relay, grp)
    return [o.detach(), *torch.autograd.grad(o, x, do.to(DEV))]


def _check(got, q, k, v, do, plan, grp, skip=()):
    o, _, _, g = O.forward_backward(q, k, v, do, plan, kv_groups=grp)
    for name, t, r in zip(("o", "dq", "dk", "dv"), got, (o, g["dq"], g["dk"], g["dv"])):
        if name in skip:
            continue
        e = rel_fro(t, r)
        say(f"  {name}: rel {e:.3e}")
        assert e <= TOL, name


@pytest.mark.parametrize("S,W,relay,D,Hq,Hkv", [
    (1, 1, False, 64, 1, 1),
    (31, 6, False, 32, 2, 2),
    (33, 32, True, 64, 2, 1),      # a window of one tile
    (65, 5, True, 128, 2, 2),
    (129, 17, True, 256, 2, 1),
    (640, 8, True, 64, 4, 2),      # 240 global rows, several query chunks
    (1300, 37, True, 128, 1, 1),
    (200, 15, False, 48, 2, 2),    # padded head dim
])
def test_edges(S, W, relay, D, Hq, Hkv):
    say(f"f32 split: S={S} W={W} relay={relay} D={D} H={Hq}/{Hkv}")
    q, k, v, do = inputs(1, Hq, Hkv, S, D, F32, seed=S + D)
    plan, grp = O.Plan(S, W, relay, 2), Hq // Hkv
    # one key: its softmax is constant, dq and dk are zero
    _check(_run(q, k, v, do, W, relay, grp), q, k, v, do, plan, grp, ("dq", "dk") if S == 1 else ())


@pytest.mark.parametrize("sv,sd", [(1e30, 1e-20), (1e-30, 1e20), (2.0 ** 100, 2.0 ** -100)])
def test_magnitudes(sv, sd):
    """V and dO far from 1 (their products stay in range)."""
    say(f"f32 split: v * {sv:g}, dO * {sd:g}")
    q, k, v, do = inputs(1, 2, 2, 300, 64, F32, seed=9)
    v, do = v * sv, do * sd
    _check(_run(q, k, v, do, 18, True, 1), q, k, v, do, O.Plan(300, 18, True, 2), 1)


def test_infinite_v():
    """A query that sees an infinite value gets that infinity; one whose tiles
    do not hold it is untouched."""
    q, k, v, do = inputs(1, 1, 1, 400, 64, F32, seed=3)
    clean = _run(q, k, v, do, 20, False, 1)[0].cpu()
    v[0, 0, 205, 7] = float("inf")
    v[0, 0, 205, 8] = float("-inf")
    o = _run(q, k, v, do, 20, False, 1)[0].cpu()
    assert bool((o[0, 0, 205:225, 7] == float("inf")).all())
    assert bool((o[0, 0, 205:225, 8] == float("-inf")).all())
    assert torch.equal(o[0, 0, :128], clean[0, 0, :128])
    keep = [d for d in range(64) if d not in (7, 8)]
    assert torch.equal(o[..., keep], clean[..., keep])
