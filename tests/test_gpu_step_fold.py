"""Row work folded into the projections (one or two rows): the same bits as the
row kernel followed by the projections, over widths at the ends of the
256-column pieces, in place and into another state."""

from __future__ import annotations

import ctypes

import pytest
import torch

from spikegpt_myelin_amd import _lib, generation
from spikegpt_myelin_amd.model import SpikeGPTConfig, SpikeLanguageModel

pytestmark = pytest.mark.gpu


def _step(model, ids, packed, fold, in_place, monkeypatch):
    monkeypatch.setattr(generation, "_FOLD_ROWS", 2 if fold else 0)
    ws = generation.StepWorkspace(*generation._model_dims(model, len(ids)), ids.device)
    src = packed.clone()
    dst = src if in_place else torch.full_like(src, float("nan"))
    for _ in range(3):  # the two residual buffers change places from step to step
        logits = generation.model_step(model, ids, src, dst, ws)
        if not in_place:
            src, dst = dst, src.fill_(float("nan"))
    torch.cuda.synchronize()
    return logits.clone(), (dst if in_place else src).clone()


@pytest.mark.parametrize("spiking", [True, False])
@pytest.mark.parametrize("in_place", [True, False])
@pytest.mark.parametrize("B,C,L", [(1, 4, 2), (1, 64, 1), (2, 100, 3), (1, 256, 2), (2, 260, 2),
                                   (1, 508, 3), (2, 768, 2), (1, 772, 2), (2, 1024, 2),
                                   (1, 1028, 2)])
def test_fold_equals_row_then_projections(B, C, L, in_place, spiking, monkeypatch):
    print(f"step fold B={B} C={C} L={L} in_place={in_place} spiking={spiking}", flush=True)
    torch.manual_seed(5)
    cfg = SpikeGPTConfig(vocab_size=61, context_length=16, n_layer=L, n_embd=C, dropout=0.0,
                         spiking=spiking)
    with torch.device("cuda"):
        model = SpikeLanguageModel(cfg).eval()
    with torch.no_grad():
        for name, p in model.named_parameters():
            if name.endswith(("key.weight", "value.weight", "receptance.weight",
                              "output.weight")):
                p.mul_(3.0)
    ids = torch.randint(0, 61, (B,), device="cuda")
    packed = torch.randn(L, 7, B, C, device="cuda")
    packed[:, 2] = packed[:, 2].abs() + 0.5
    plain = _step(model, ids, packed, False, in_place, monkeypatch)
    fold = _step(model, ids, packed, True, in_place, monkeypatch)
    assert torch.equal(plain[1], fold[1])
    assert torch.equal(plain[0], fold[0])
    assert bool(torch.isfinite(fold[0]).all())


def test_fold_argument_errors():
    lib = _lib.load()
    r, a = _lib.StepRowArgs(), _lib.StepLinearArgs()
    t = torch.zeros(64, 64, device="cuda")
    a.batch, a.k, a.n0, a.n1 = 2, 16, 16, 16
    a.w[0] = a.w[1] = t.data_ptr()
    a.out[0], a.out[1] = t[40].data_ptr(), t[48].data_ptr()
    r.batch, r.channels, r.n_mix = 2, 16, 2
    for j, name in enumerate(("add", "membrane_in", "residual", "ln_weight", "ln_bias",
                              "previous_in", "membrane_out", "previous_out")):
        setattr(r, name, t[8 + j].data_ptr())
    r.mix[0] = r.mix[1] = t[0].data_ptr()
    new = t[30].data_ptr()

    def call(mode=2, out=new):
        return lib.block_step_row_linear(mode, ctypes.byref(r), out, ctypes.byref(a),
                                         torch.cuda.current_stream().cuda_stream)

    assert call() == 0
    assert call(mode=0) == 1 and call(mode=3) == 1
    assert call(out=None) == 1
    assert call(out=r.residual) == 1  # overlaps what other workgroups read
    r.previous_out = r.previous_in + 64
    assert call() == 1
    r.previous_out = t[15].data_ptr()
    r.batch = a.batch = 3
    assert call() == 1
    r.batch = a.batch = 2
    r.channels = a.k = 1028
    assert call() == 1
    a.batch, a.k = 1, 16
    a.x[0] = t.data_ptr()
    assert lib.block_step_linear_copy(ctypes.byref(a), None, new, new, 4, None) == 1
    torch.cuda.synchronize()
