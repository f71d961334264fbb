"""fp32 on the bf16 matrix core (every operand cut in three bf16 pieces): tile
edges against the fp64 oracle with the fp32 tolerances, single products with the
bits that cost a split most, inputs far from 1, and infinite inputs.

Tolerances: relative Frobenius 2e-6 of o and the gradients. The three left-out
piece products are at most 2^-24 of a product, an fp32 accumulation over n
terms adds about sqrt(n) 2^-24 (n <= 1300 keys or queries here): 6e-8 +
36 * 6e-8 = 2.2e-6 at most, and all measured below 6e-7. Where n is larger the
tolerance grows with sqrt(n)."""
import math

import pytest
import torch

import cron_root_attention as cra
from cron_root_attention import _native
from cron_root_attention.core import _attention_with_plan
from oracle import cra_oracle as O
from tests.parity_util import DEV, F32, inputs, rel_fro, say

pytestmark = pytest.mark.gpu
TOL = 2e-6


def _run(q, k, v, do, W, relay, grp):
    x = [t.to(DEV).requires_grad_(True) for t in (q, k, v)]
    o = _attention_with_plan(*x, W, relay, grp)
    return [o.detach(), *torch.autograd.grad(o, x, do.to(DEV))]


def _check(got, q, k, v, do, plan, grp, skip=(), tol=TOL):
    o, _, _, g = O.forward_backward(q, k, v, do, plan, kv_groups=grp)
    for name, t, r in zip(("o", "dq", "dk", "dv"), got, (o, g["dq"], g["dk"], g["dv"])):
        if name in skip:
            continue
        e = rel_fro(t, r)
        say(f"  {name}: rel {e:.3e}")
        assert e <= tol, name


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


@pytest.mark.parametrize("W,Hq,Hkv,D", [(400, 32, 1, 64), (650, 16, 2, 128)])
def test_long_local_sums(W, Hq, Hkv, D):
    """Grouped heads and a wide window: a key row sums over W queries of each
    head of its group (12800 and 5200 here)."""
    say(f"f32 split: W={W} D={D} H={Hq}/{Hkv}")
    q, k, v, do = inputs(1, Hq, Hkv, 1300, D, F32, seed=W)
    grp = Hq // Hkv
    _check(_run(q, k, v, do, W, True, grp), q, k, v, do, O.Plan(1300, W, True, 2), grp,
           tol=TOL * math.sqrt(W * grp / 1300))


@pytest.mark.parametrize("low", [0xffff, 0x7fff, 0x8001, 0x7f7f, None])
def test_products(low):
    """The log-sum-exp of one key is its score: 32 equal products q k of one
    sign, with given low bits of the significands, in fp32 steps of known
    error: left-out pieces 2^-24, the sum's last rounding 2^-23 (the matrix
    core may cut it off), the roundings of s * log2(e) / sqrt(D) and of its
    product with ln 2, 2^-24 each: 2.5 * 2^-23 = 3e-7. Pieces cut off instead
    of rounded leave 2^-21 = 4.7e-7 for 0xffff."""
    H = 512
    g = torch.Generator().manual_seed(7)

    def bits():
        n = low
        if n is None:
            n = torch.randint(0, 1 << 16, (1, H, 1, 1), generator=g, dtype=torch.int32)
        return (torch.full((1, H, 1, 1), 0x3f800000, dtype=torch.int32) | n).view(F32)

    q, k = (bits().expand(1, H, 1, 32).contiguous() for _ in range(2))
    p = _native.problem(1, H, H, 1, 32, 1, False, 2, F32, 1 / math.sqrt(32))
    qd, kd, none = q.to(DEV), k.to(DEV), torch.zeros(1, H, 1, 32, device=DEV)
    _, lse = _native.forward(p, qd, kd, none, none, none, phases=_native.PHASE_LOCAL)
    c2 = torch.tensor(1 / math.sqrt(32), dtype=F32) * torch.tensor(math.log2(math.e), dtype=F32)
    want = (q.double() * k.double()).sum(-1)[..., 0] * c2.double()
    want *= torch.tensor(math.log(2), dtype=F32).double()
    e = float((lse[..., 0].cpu().double() / want[0] - 1).abs().max())
    say(f"f32 split: low bits {low and hex(low)}: {e:.2e}")
    assert e <= 3e-7


@pytest.mark.parametrize("D", [32, 256])
def test_largest_floats(D):
    """Finite values that round to infinity in bf16 stay what they are (one key:
    o = v), and infinities and NaN too, next to each other."""
    top = torch.finfo(F32).max
    x = torch.tensor([top, -top, 3.3961775e38, 3.39e38, math.inf, -math.inf, math.nan, 1.5])
    v = x.repeat(D // 8).view(1, 1, 1, D)
    q, k = (torch.ones(1, 1, 1, D) for _ in range(2))
    with torch.no_grad():
        o = cra.cron_root_attention(*(t.to(DEV) for t in (q, k, v))).cpu()
    assert torch.equal(o.isnan(), v.isnan())
    ok = ~v.isnan()
    assert torch.equal(o[ok], v[ok])


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
