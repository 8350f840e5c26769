"""Key, value and receptance as tiles of their own and the WKV kernel after them:
the same bits as the tile that ends in the update, at the edges of the rule."""

from __future__ import annotations

import pytest
import torch

from spikegpt_myelin_amd import generation
from spikegpt_myelin_amd.model import SpikeGPTConfig, SpikeLanguageModel

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("B,C", [(5, 512), (16, 516), (17, 640), (33, 768), (48, 768), (80, 512), (32, 1024)])
def test_apart_equals_one_tile(B, C, monkeypatch):
    print(f"step apart B={B} C={C}", flush=True)
    assert generation._apart(B, C) and generation._own_linear(B, C)
    torch.manual_seed(3)
    cfg = SpikeGPTConfig(vocab_size=61, context_length=16, n_layer=2, n_embd=C, dropout=0.0)
    with torch.device("cuda"):
        model = SpikeLanguageModel(cfg).eval()
    ids = torch.randint(0, 61, (B,), device="cuda")
    packed = torch.randn(2, 7, B, C, device="cuda")
    packed[:, 2] = packed[:, 2].abs() + 0.5
    got = []
    for apart in (False, True):
        monkeypatch.setattr(generation, "_apart", lambda b, c, apart=apart: apart)
        ws = generation.StepWorkspace(*generation._model_dims(model, B), ids.device)
        state = packed.clone()
        got.append((generation.model_step(model, ids, state, state, ws).clone(), state))
    torch.cuda.synchronize()
    assert torch.equal(got[0][0], got[1][0]) and torch.equal(got[0][1], got[1][1])


def test_rule():
    assert not generation._apart(4, 768) and not generation._apart(16, 256)
    assert not generation._apart(64, 768) and not generation._apart(128, 512)
