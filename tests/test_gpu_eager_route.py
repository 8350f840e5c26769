"""Plain eager calls of the activations, mixes and RWKV-7 run over the same
launchers as the custom ops: same values and gradients bit for bit, and calls
under a dispatch mode, a transform or a forward-mode level keep the op route."""

from __future__ import annotations

import pytest
import torch
from torch.utils._python_dispatch import TorchDispatchMode

from spikegpt_myelin_amd import gates, lif, timemix, wkv, wkv7

pytestmark = pytest.mark.gpu
DEV = torch.device("cuda", 0)


class _Seen(TorchDispatchMode):
    def __init__(self):
        super().__init__()
        self.names = set()

    def __torch_dispatch__(self, func, types, args=(), kwargs=None):
        self.names.add(str(func))
        return func(*args, **(kwargs or {}))


def _calls():
    g = torch.Generator(device=DEV).manual_seed(0)

    def rand(*shape, dtype=torch.float32):
        return torch.randn(*shape, device=DEV, generator=g).to(dtype)

    bf = torch.bfloat16
    norm = torch.nn.LayerNorm(256).to(DEV)
    w = torch.rand(2, 9, 1, 64, device=DEV, generator=g)
    return {
        "lif": (lambda x: lif.lif_sequence(x), [rand(2, 70, 24, dtype=bf)]),
        "lif_residual": (lambda r, x: lif.lif_residual(r, x), [rand(2, 70, 24),
                                                              rand(2, 70, 24, dtype=bf)]),
        "relu_square": (lambda x: gates.relu_square(x), [rand(3, 40, dtype=bf)]),
        "sigmoid_gate": (lambda r, x: gates.sigmoid_gate(r, x), [rand(3, 40, dtype=bf),
                                                                 rand(3, 40, dtype=bf)]),
        "shift_mix": (lambda x, m: timemix.token_shift_mix(x, m), [rand(2, 9, 40), rand(3, 40)]),
        "ln_fork": (lambda x, m: timemix.layer_norm_shift_mix_fork(x, norm, m),
                    [rand(2, 9, 256), rand(2, 256)]),
        "ln_mix": (lambda x, m: timemix.layer_norm_shift_mix(x, norm, m),
                   [rand(2, 9, 256), rand(3, 256)]),
        "wkv": (lambda *a: wkv.weighted_key_value_hip(*a), [rand(2, 9, 40), rand(2, 9, 40),
                                                            rand(40), rand(40)]),
        "wkv7": (lambda *a: wkv7.wkv7_forward(*a),
                 [rand(2, 9, 1, 64), w, *(0.1 * rand(2, 9, 1, 64) for _ in range(4)),
                  rand(2, 1, 64, 64)]),
    }


def _flat(out):
    return list(out) if isinstance(out, (tuple, list)) else [out]


@pytest.mark.parametrize("name", ["lif", "lif_residual", "ln_fork", "ln_mix", "relu_square",
                                  "shift_mix", "sigmoid_gate", "wkv", "wkv7"])
def test_eager_route_equals_op_route(name):
    fn, inputs = _calls()[name]
    print(f"eager route {name}", flush=True)
    results = []
    for mode in (False, True):
        leaves = [t.clone().requires_grad_() for t in inputs]
        seen = _Seen()
        if mode:
            with seen:
                outs = _flat(fn(*leaves))
        else:
            outs = _flat(fn(*leaves))
        g = torch.Generator(device=DEV).manual_seed(1)
        grads = [torch.randn(o.shape, device=DEV, generator=g).to(o.dtype) for o in outs]
        got = torch.autograd.grad(outs, leaves, grads)
        # only the first output used: the others' gradients are absent
        leaves2 = [t.clone().requires_grad_() for t in inputs]
        first = _flat(fn(*leaves2))[0]
        got2 = torch.autograd.grad(first, leaves2, grads[0], allow_unused=True)
        results.append((outs, got, got2))
        if mode:
            assert any("myelin" in n for n in seen.names), seen.names
    for a, b in zip(*results):
        for x, y in zip(a, b):
            assert (x is None) == (y is None)
            if x is not None:
                assert x.dtype == y.dtype and torch.equal(x, y)
    with torch.no_grad():  # calls that save nothing
        for x, y in zip(_flat(fn(*inputs)), results[0][0]):
            assert torch.equal(x, y)


def test_saved_tensor_hooks_see_what_is_saved():
    packed = []
    x = torch.randn(2, 40, 24, device=DEV).bfloat16().requires_grad_()
    with torch.autograd.graph.saved_tensors_hooks(lambda t: packed.append(t.shape) or t.clone(),
                                                  lambda t: t):
        y = lif.lif_sequence(gates.relu_square(x))
    assert len(packed) >= 3
    (gx,) = torch.autograd.grad(y.float().sum(), x)
    assert gx.shape == x.shape


def test_in_place_change_of_a_saved_input_is_refused():
    r = torch.randn(3, 40, device=DEV).bfloat16().requires_grad_()
    x = torch.randn(3, 40, device=DEV).bfloat16()
    y = gates.sigmoid_gate(r, x)
    x.add_(1)
    with pytest.raises(RuntimeError, match="modified by an inplace operation"):
        y.float().sum().backward()
