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


class _Doubled(torch.nn.Module):
    """A parametrisation: the weight is computed on each access."""

    def forward(self, w):
        return 2.0 * w


@pytest.mark.gpu
@pytest.mark.parametrize("change", ["eps", "activation", "shape", "transposed", "parametrised"])
def test_the_record_follows_what_it_was_made_from(change):
    """A changed normaliser eps or activation, a weight of another shape or layout at the same address, weights computed
    on access: the one-launch forward gives what the layers give."""
    m = _model(width=32, hidden=(32, 16)).to("cuda")
    obs = {"g": torch.randn(100, 32, device="cuda")}
    with torch.no_grad():
        before = m(obs)
        if change == "eps":
            m.obs_normalizer.eps = 0.5
        elif change == "activation":
            m.act_code = L.ACTIVATIONS["tanh"]
        elif change == "shape":  # the same memory as another layer stack: 32 -> 16 -> 16 -> 4
            first, second = m.mlp[0], m.mlp[2]
            first.weight.data = first.weight.data[:16]
            first.bias.data = first.bias.data[:16]
            second.weight.data = second.weight.data.view(-1)[:256].view(16, 16)
            first.out_features, second.in_features = 16, 16
        elif change == "transposed":  # (the layers take contiguous weights only)
            m.mlp[0].weight.data = m.mlp[0].weight.data.t()
            for call in (m, m.forward_layers):
                with pytest.raises(ValueError, match="contiguous"):
                    call(obs)
            return
        elif change == "parametrised":
            torch.nn.utils.parametrize.register_parametrization(m.mlp[2], "weight", _Doubled())
        else:
            m.mlp[0].weight.data = m.mlp[0].weight.data.clone()
        after, want = m(obs), m.forward_layers(obs)
        assert float((after - want).norm() / want.norm()) < 1e-5
        assert not torch.equal(before, after)
        for _ in range(20):  # (memory handed round between the computed weights, the output and the workspace)
            assert torch.equal(m(obs), after)
