"""Layer norm + token-shift mixes for rows of other widths (the row-spread
kernels behind layer_norm_shift_mix): edges of a wave's 256 channels and of a
4-row batch, against F.layer_norm and the oracle's mix in float64."""

from __future__ import annotations

import pytest
import torch
import torch.nn.functional as F

from oracle import timemix as TM
from spikegpt_myelin_amd.timemix import layer_norm_shift_mix, layer_norm_shift_mix_fork

pytestmark = pytest.mark.gpu
DEV = torch.device("cuda", 0)


def _reference(x, w, b, mix, eps=1e-5):
    y = F.layer_norm(x, (x.shape[-1],), w, b, eps)
    return [TM.mix_with_previous(y, mix[j]) for j in range(mix.shape[0])]


# C: one lane, a partial wave, two, three and four waves with and without a
# tail; T: 1, a batch and its neighbours, a chunk of 16 rows and its neighbours.
@pytest.mark.parametrize("B,T,C,n", [(1, 1, 4, 2), (2, 3, 64, 3), (3, 4, 136, 2), (2, 5, 252, 3),
                                     (1, 15, 260, 3), (2, 16, 640, 2), (3, 17, 768, 3),
                                     (1, 131, 1020, 3), (2, 33, 1024, 2)])
@pytest.mark.parametrize("dtype", [torch.float32, torch.bfloat16, torch.float16])
@pytest.mark.parametrize("fork", [True, False])
def test_rows_match_layer_norm_then_mix(B, T, C, n, dtype, fork):
    print(f"ln rows B={B} T={T} C={C} n={n} {dtype} fork={fork}", flush=True)
    g = torch.Generator().manual_seed(B * 1000 + T + C)
    x = torch.randn(B, T, C, generator=g) * 2 + 0.5
    w = 1 + 0.3 * torch.randn(C, generator=g)
    b = 0.2 * torch.randn(C, generator=g)
    mix = torch.rand(n, C, generator=g)
    grads = [torch.randn(B, T, C, generator=g).to(dtype) for _ in range(n)]
    res = torch.randn(B, T, C, generator=g)
    xd, wd, bd, md = (t.double().requires_grad_() for t in (x, w, b, mix))
    ref = _reference(xd, wd, bd, md)
    torch.autograd.backward(ref + ([xd * 1.0] if fork else []),
                            [t.double() for t in grads] + ([res.double()] if fork else []))
    norm = torch.nn.LayerNorm(C).to(DEV)
    with torch.no_grad():
        norm.weight.copy_(w)
        norm.bias.copy_(b)
    xg, mg = x.to(DEV).requires_grad_(), mix.to(DEV).requires_grad_()
    fn = layer_norm_shift_mix_fork if fork else layer_norm_shift_mix
    if dtype == torch.float32:
        outs = fn(xg, norm, mg)
    else:
        with torch.autocast("cuda", dtype=dtype):
            outs = fn(xg, norm, mg)
    gpu = [t.to(DEV) for t in grads]
    if fork:
        assert outs[-1].data_ptr() == xg.data_ptr()
        gpu.append(res.to(DEV))
    torch.autograd.backward(outs, gpu)
    # fp32: the sums of C <= 1024 products of order one; 16 bits: one rounding
    # (unit roundoff 2^-8 for bf16's 8 significant bits, 2^-11 for fp16's 11).
    tol = {torch.float32: 2e-5, torch.bfloat16: 2.0 ** -8, torch.float16: 2.0 ** -11}[dtype]
    for o, r in zip(outs[:n], ref):
        assert o.dtype == dtype
        torch.testing.assert_close(o.cpu().double(), r.detach(), atol=2e-5, rtol=tol + 2e-5)
    for got, want, name in ((xg.grad, xd.grad, "x"), (norm.weight.grad, wd.grad, "weight"),
                            (norm.bias.grad, bd.grad, "bias"), (mg.grad, md.grad, "mix")):
        scale = want.abs().max().item() + 1e-12
        err = (got.cpu().double() - want).abs().max().item() / scale
        assert err < 2e-5, f"grad {name}: {err:.2e} of {scale:.3g}"


def test_hooks_and_frozen_parameters_keep_working():
    # A hooked layer norm takes the unfused route (its hook runs); outputs that
    # are not used get no gradient.
    x = torch.randn(2, 9, 96, device=DEV, requires_grad=True)
    norm = torch.nn.LayerNorm(96).to(DEV)
    mix = torch.rand(2, 96, device=DEV)
    plain = layer_norm_shift_mix(x, norm, mix)
    seen = []
    handle = norm.register_forward_hook(lambda m, i, o: seen.append(1))
    hooked = layer_norm_shift_mix(x, norm, mix)
    handle.remove()
    assert seen
    for a, b in zip(plain, hooked):
        torch.testing.assert_close(a, b, atol=1e-5, rtol=1e-5)
    (ga,) = torch.autograd.grad(plain[1].sum(), x)
    (gb,) = torch.autograd.grad(hooked[1].sum(), x)
    torch.testing.assert_close(ga, gb, atol=1e-5, rtol=1e-5)
