"""The layers' form of the op (output and gradients as views of [B, S, H, D]
buffers): the op's values bit for bit, in the layout that the projections take."""
import pytest
import torch

import cron_root_attention as cra
from cron_root_attention.core import _layer_attention
from tests.parity_util import BF16, DEV, F16, F32, inputs

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("B,Hq,Hkv,S,D,dtype", [
    (1, 4, 4, 1, 64, F16),
    (2, 6, 3, 300, 128, BF16),
    (1, 4, 1, 2500, 64, F16),     # relay
    (2, 2, 1, 200, 256, BF16),
    (1, 2, 2, 333, 64, F32),
    (1, 2, 2, 100, 80, F16),      # padded head dim: the op's own output
])
def test_values_and_layout(B, Hq, Hkv, S, D, dtype):
    q, k, v, do = (t.to(DEV).transpose(1, 2).contiguous().transpose(1, 2)
                   for t in inputs(B, Hq, Hkv, S, D, dtype, seed=S))
    x = [t.requires_grad_(True) for t in (q, k, v)]
    o = cra.cron_root_attention(*x, kv_groups=Hq // Hkv)
    want = torch.autograd.grad(o, x, do)
    assert o.is_contiguous()
    with torch.no_grad():
        assert torch.equal(_layer_attention(*x, kv_groups=Hq // Hkv), o)
    y = _layer_attention(*x, kv_groups=Hq // Hkv)
    got = torch.autograd.grad(y, x, do)
    assert torch.equal(y, o)
    for a, b in zip(got, want):
        assert torch.equal(a, b)
    if D != 80:
        for t in (y, *got):
            assert t.transpose(1, 2).is_contiguous()


def _layers():
    yield "CronRootAttention", cra.CronRootAttention(256, 4, n_kv_heads=2), "o_proj"
    yield "CronRootAttentionHybrid", cra.CronRootAttentionHybrid(256, 4, threshold=1), "o_proj"
    yield "CronRootMultiheadAttention", cra.CronRootMultiheadAttention(256, 4), "out_proj"


@pytest.mark.parametrize("how", ["pre-hook", "hook", "module", "global pre-hook"])
def test_output_edited_in_place(how):
    """What a hook or module on the output projection does to its input in place
    is for the layer's copy: the backward reads the attention output."""
    for name, layer, proj in _layers():
        torch.manual_seed(0)
        layer = layer.to(DEV, F16)
        lin = getattr(layer, proj)
        lin.requires_grad_(how != "hook")  # (the linear's weight gradient reads its input)
        x = torch.randn(1, 300, 256, device=DEV, dtype=F16)
        dy = torch.randn_like(x)

        def step():
            y = x.clone().requires_grad_(True)
            out = layer(y, y, y)[0] if name == "CronRootMultiheadAttention" else layer(y)
            return [out.detach(), *torch.autograd.grad(out, y, dy)]

        def edit(m, args, *_):
            if m is lin:
                args[0].mul_(2)

        def copy(m, args):
            return (args[0] * 2,)

        if how == "hook":  # after the product: the result is the layer's own
            want = step()
            lin.register_forward_hook(edit)
            got = step()
        else:
            h = lin.register_forward_pre_hook(copy)
            want = step()
            h.remove()
            if how == "pre-hook":
                lin.register_forward_pre_hook(edit)
                got = step()
            elif how == "global pre-hook":
                h = torch.nn.modules.module.register_module_forward_pre_hook(edit)
                got = step()
                h.remove()
            else:
                class Twice(torch.nn.Module):
                    def forward(self, t):
                        return t.mul_(2)

                setattr(layer, proj, torch.nn.Sequential(Twice(), lin))
                got = step()
        for a, b in zip(got, want):
            assert torch.equal(a, b), name


def test_layer_gradients_reach_fused_projections():
    """CronRootMultiheadAttention: q, k, v are slices of one projection."""
    torch.manual_seed(0)
    m = cra.CronRootMultiheadAttention(128, 2).to(DEV, F16)
    x = torch.randn(1, 257, 128, device=DEV, dtype=F16, requires_grad=True)
    y, _ = m(x, x, x)
    dy = torch.randn_like(y)
    got = torch.autograd.grad(y, [x, m.in_proj_weight, m.in_proj_bias], dy)
    qkv = torch.nn.functional.linear(x, m.in_proj_weight, m.in_proj_bias)
    q, k, v = (t.transpose(1, 2) for t in qkv.view(1, 257, 3, 2, 64).unbind(2))
    o = cra.cron_root_attention(q, k, v).transpose(1, 2).reshape(1, 257, 128)
    want = torch.autograd.grad(m.out_proj(o), [x, m.in_proj_weight, m.in_proj_bias], dy)
    for a, b in zip(got, want):
        assert torch.allclose(a.float(), b.float(), rtol=2e-3, atol=2e-3 * float(b.abs().max()))
