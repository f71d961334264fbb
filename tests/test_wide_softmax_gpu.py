"""Softmax of the fp16/bf16 forward at head dim 256: the maximum is raised with
every 32-key tile, P is rounded for P.V only, l sums the unrounded P. Checked
against the same steps in torch fp32, where nothing but the order of fp32 sums
differs.

Tolerances: an fp32 sum of n terms is off by about sqrt(n) 2^-24 of them (n =
256 for a score of magnitude up to 8, 96 keys for l): 1e-5 for the log-sum-exp.
O differs where such an error moves a P or an O across a rounding boundary, for
about one element in 2000 by one unit in the last place (2^-7 of a bf16, 2^-10
of an fp16): relative 2^-7 / sqrt(2000) = 1.7e-4. A P rounded relative to
another maximum, or an l of rounded P, is another rounding of every element:
2e-3 in bf16, 2.5e-4 in fp16, and up to 2e-3 and 2e-4 in the log-sum-exp."""
import math

import pytest
import torch

from cron_root_attention import _native
from tests.parity_util import BF16, DEV, F16, inputs, rel_fro, say

pytestmark = pytest.mark.gpu


def _steps(q, k, v, W):
    """Sliding window of W keys, the tiles of 64-query workgroups."""
    S, D = q.shape
    dt = q.dtype
    s = (q.float() @ k.float().t()) * (math.log2(math.e) / math.sqrt(D))
    i = torch.arange(S)[:, None]
    see = (torch.arange(S)[None] <= i) & (torch.arange(S)[None] > i - W)
    s = s.masked_fill(~see, -math.inf)
    o, lse = torch.zeros(S, D), torch.zeros(S)
    for m0 in range(0, S, 64):
        hi = min(S, m0 + 64)
        m = torch.full((hi - m0,), -math.inf)
        l, acc = torch.zeros(hi - m0), torch.zeros(hi - m0, D)
        for t in range(max(0, m0 - W + 1), hi, 32):
            x = s[m0:hi, t:min(t + 32, hi)]
            new = torch.maximum(m, x.max(1).values)
            use = new.masked_fill(new == -math.inf, 0.)
            a, p = torch.exp2(m - use), torch.exp2(x - use[:, None])
            l = l * a + p.sum(1)
            acc = acc * a[:, None] + p.to(dt).float() @ v[t:min(t + 32, hi)].float()
            m = new
        o[m0:hi], lse[m0:hi] = acc / l[:, None], (m + torch.log2(l)) * math.log(2)
    return o.to(dt), lse


@pytest.mark.parametrize("dtype", [F16, BF16])
@pytest.mark.parametrize("S,W", [(33, 33), (96, 96), (200, 37), (300, 64)])
def test_steps(S, W, dtype):
    say(f"wide softmax: S={S} W={W} {dtype}")
    q, k, v, _ = inputs(1, 1, 1, S, 256, dtype, seed=S)
    v += 1  # an O away from 0, so that the normaliser counts
    p = _native.problem(1, 1, 1, S, 256, W, False, 2, dtype, 1 / 16)
    none = torch.zeros(1, 1, (S + W - 1) // W, 256, dtype=dtype, device=DEV)
    qd, kd, vd = (t.to(DEV) for t in (q, k, v))
    o, lse = _native.forward(p, qd, kd, vd, none, none, phases=_native.PHASE_LOCAL)
    want, want_lse = _steps(q[0, 0], k[0, 0], v[0, 0], W)
    e = float((lse[0, 0].cpu() - want_lse).abs().max())
    r = rel_fro(o[0, 0], want.double())
    say(f"  lse {e:.2e}, o rel {r:.2e}")
    assert e <= 1e-5
    assert r <= (1.7e-4 if dtype == BF16 else 2.2e-5)
