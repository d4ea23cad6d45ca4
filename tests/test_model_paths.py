"""MLPModel's shortcuts (the one-launch forward, its record, the layered bootstrap forward) against what calling the model
does: copies, hooks, overrides, changed and computed parameters."""

from __future__ import annotations

import copy
import io
import pickle

import pytest
import torch

from tt_rsl_rl_amd import _lib as L
from tt_rsl_rl_amd import models
from tt_rsl_rl_amd.models import MLPModel


def _model(cls=MLPModel, width=20, out=4, hidden=(32, 16), norm=True, **kw):
    torch.manual_seed(0)
    return cls({"g": torch.zeros(2, width)}, {"critic": ["g"]}, "critic", out, hidden_dims=list(hidden), activation="elu",
               obs_normalization=norm, **kw)


def _copies(m):
    saved = io.BytesIO()
    torch.save(m, saved)
    saved.seek(0)
    return [copy.deepcopy(m), copy.copy(m), pickle.loads(pickle.dumps(m)), torch.load(saved, weights_only=False)]


def test_a_model_with_a_record_copies_and_pickles():
    m = _model()
    rec = L.MlpProblem(num_layers=3)
    rec.layers[0] = L.MlpLayer(4096, 8192, 20, 32)
    m._fused = models._FusedRecord(((4096, 8192), rec, 0))
    for c in _copies(m):
        assert c._fused is None or c is m or c._fused is m._fused
        assert all(torch.equal(a, b) for a, b in zip(m.parameters(), c.parameters(), strict=True))
    assert copy.deepcopy(m)._fused is None and pickle.loads(pickle.dumps(m))._fused is None


@pytest.mark.gpu
def test_a_model_that_ran_copies_and_pickles():
    m = _model().to("cuda")
    obs = {"g": torch.randn(50, 20, device="cuda")}
    with torch.no_grad():
        y = m(obs)
        assert m._fused is not None and m._fused[1] is not None
        for c in _copies(m):
            assert torch.equal(c(obs), y)
