"""Global-row dK/dV at the edges of its geometries: the packed rows on either
side of the limit between the 64-row and the wide workgroups, and packed
documents whose lengths sit at the edges of a query chunk.

A small window gives many packed rows at few tokens (rows = ceil(S / W) * 3
with relay), so the fp64 oracle covers every gradient in full. Tolerance: the
gradient tolerance of the parity tests (relative Frobenius, 1e-2 fp16 and
3e-2 bf16: P and dS are rounded to the input type, 2^-11 and 2^-8)."""
import pytest
import torch

from cron_root_attention.core import _attention_with_plan, _varlen_with_plan
from oracle import cra_oracle as O
from tests.parity_util import BF16, DEV, F16, F32, TOL_GRAD, inputs, rel_fro, say

pytestmark = pytest.mark.gpu


def _check(grads, ref, dtype):
    for name, t in zip(("dq", "dk", "dv"), grads):
        e = rel_fro(t, ref[name])
        say(f"  {name}: rel {e:.3e}")
        assert e <= TOL_GRAD[dtype], name


@pytest.mark.parametrize("S,W,D,Hq,Hkv,dtype", [
    (2048, 8, 128, 2, 2, F16),    # 768 rows: the last 64-row problem of few workgroups
    (2049, 8, 128, 2, 2, F16),    # 771 rows: 192-row workgroups
    (700, 11, 128, 4, 2, BF16),   # 192 rows, grouped heads: three full 64-row tiles
    (2048, 8, 64, 2, 2, F16),     # 768 rows below D = 128
    (2049, 8, 64, 2, 1, BF16),    # 771 rows below D = 128: 128-row workgroups
    (300, 9, 128, 256, 256, F16),  # 102 rows, two wide workgroups per CU: 192-row workgroups
    (400, 20, 128, 128, 64, F16), # 60 rows: one 64-row tile
    (330, 19, 64, 8, 1, F16),     # grouped heads: chunks of 64 queries, the last of 10
    (256, 16, 128, 16, 2, BF16),  # grouped heads: exact chunks of 64 queries
    (300, 9, 64, 256, 256, F16),  # more 128-key local workgroups than CUs
    (129, 12, 32, 512, 256, BF16),
    (129, 12, 64, 4, 1, F16),     # fewer: 64-key ones, the last of one key
    (65, 65, 32, 1, 1, F16),      # one block: no query sees a global row
])
def test_row_limits(S, W, D, Hq, Hkv, dtype):
    say(f"global rows: S={S} W={W} D={D} H={Hq}/{Hkv} {dtype}")
    q, k, v, do = inputs(1, Hq, Hkv, S, D, dtype, seed=S + D)
    plan = O.Plan(S, W, True, 2)
    _, _, _, ref = O.forward_backward(q, k, v, do, plan, kv_groups=Hq // Hkv)
    x = [t.to(DEV).requires_grad_(True) for t in (q, k, v)]
    o = _attention_with_plan(*x, W, True, Hq // Hkv)
    _check(torch.autograd.grad(o, x, do.to(DEV)), ref, dtype)


@pytest.mark.parametrize("D,dtype,lens", [
    (128, F16, (1, 63, 64, 65, 127, 128, 129, 640)),
    (64, BF16, (513, 1, 1, 64, 192, 65)),
])
def test_document_chunks(D, dtype, lens):
    """Chunks of one length over all documents (64 queries here): documents
    of a part of a chunk, exact chunks and one query more."""
    say(f"document chunks: D={D} {dtype} lens={lens}")
    S = sum(lens)
    cu = [0]
    for n in lens:
        cu.append(cu[-1] + n)
    W = [max(1, min(n, 5)) for n in lens]
    relay = [n >= 64 for n in lens]
    q, k, v, do = inputs(1, 4, 2, S, D, dtype, seed=S)
    x = [t.to(DEV).requires_grad_(True) for t in (q, k, v)]
    o = _varlen_with_plan(*x, cu, W, relay, kv_groups=2)
    got = torch.autograd.grad(o, x, do.to(DEV))
    for i, (a, b) in enumerate(zip(cu, cu[1:])):
        part = [t[:, :, a:b] for t in (q, k, v, do)]
        _, _, _, ref = O.forward_backward(*part, O.Plan(b - a, W[i], relay[i], 2), kv_groups=2)
        if b - a == 1:  # one key: its softmax is constant, dq and dk are zero
            assert rel_fro(got[2][:, :, a:b], ref["dv"]) <= TOL_GRAD[dtype]
            continue
        _check([t[:, :, a:b] for t in got], ref, dtype)


@pytest.mark.parametrize("D,dtype,H,W,lens", [
    (64, F16, 8, 2, (1100, 530, 270)),        # chunks of 256, 192 and 192 queries
    (64, F32, 12, 2, (1000, 300, 260, 1)),    # 256, 192, 192 and one
    (128, BF16, 16, 9, (70,) * 90),           # uncut, two launches of documents
])
def test_documents_cut_evenly(D, dtype, H, W, lens):
    """Each document in chunks of its own even length, or none cut."""
    say(f"documents cut evenly: D={D} {dtype} H={H} W={W} lens={lens[:4]}")
    S = sum(lens)
    cu = [0]
    for n in lens:
        cu.append(cu[-1] + n)
    Ws = [min(n, W) for n in lens]
    relay = [n >= 64 for n in lens]
    q, k, v, do = inputs(1, H, H, S, D, dtype, seed=S)
    x = [t.to(DEV).requires_grad_(True) for t in (q, k, v)]
    o = _varlen_with_plan(*x, cu, Ws, relay)
    got = torch.autograd.grad(o, x, do.to(DEV))
    for i, (a, b) in list(enumerate(zip(cu, cu[1:])))[::max(1, len(lens) // 8)]:
        part = [t[:, ::5, a:b] for t in (q, k, v, do)]
        _, _, _, ref = O.forward_backward(*part, O.Plan(b - a, Ws[i], relay[i], 2))
        if b - a > 1:
            _check([t[:, ::5, a:b] for t in got], ref, dtype)
