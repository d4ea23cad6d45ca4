"""The one-launch MLP forward (ppo_mlp_fwd) against the layers in fp64 and against the layer-by-layer path.  Tolerance: the
fp32 GEMMs' bar per layer (2e-6 of the result's norm), times the layers."""

from __future__ import annotations

import pytest
import torch

from tt_rsl_rl_amd import models
from tt_rsl_rl_amd.models import MLPModel

pytestmark = pytest.mark.gpu


def _model(widths, actions, hidden, act, norm, seed=0):
    torch.manual_seed(seed)
    obs = {f"g{i}": torch.zeros(2, w) for i, w in enumerate(widths)}
    m = MLPModel(obs, {"actor": list(obs)}, "actor", actions, hidden_dims=hidden, activation=act, obs_normalization=norm,
                 distribution_cfg=dict(class_name="GaussianDistribution")).to("cuda")
    if norm:
        m.obs_normalizer._mean.copy_(torch.randn_like(m.obs_normalizer._mean))
        m.obs_normalizer._std.copy_(torch.rand_like(m.obs_normalizer._std) + 0.1)
    return m


def _exact(m, obs):
    x = torch.cat([obs[g] for g in m.obs_groups], -1).double()
    if m.obs_normalization:
        x = (x - m.obs_normalizer._mean.double()) / (m.obs_normalizer._std.double() + m.obs_normalizer.eps)
    for layer in m.mlp:
        x = torch.nn.functional.linear(x, layer.weight.double(), layer.bias.double()) \
            if isinstance(layer, torch.nn.Linear) else layer(x)
    return x


# rows around the 16-row blocks; widths around the 16-wide tiles and k-groups, with and without 16-byte rows; one layer's
# tiles on every wave, on few, on several rounds
@pytest.mark.parametrize("rows", [1, 15, 16, 17, 333, 4096])
@pytest.mark.parametrize("widths,actions,hidden", [((48,), 12, [512, 256, 128]), ((96, 3), 29, [512, 256, 128]),
                                                   ((1,), 1, [4]), ((17, 16), 40, [33, 130]), ((235,), 3, [400, 200, 100]),
                                                   ((64,), 16, [1024, 16, 1024])])
def test_forward_matches_fp64(rows, widths, actions, hidden):
    for act, norm in (("elu", True), ("tanh", False), ("relu", True)):
        m = _model(widths, actions, hidden, act, norm)
        obs = {f"g{i}": torch.randn(rows, w + 3, device="cuda")[:, 1:w + 1] for i, w in enumerate(widths)}
        with torch.inference_mode():
            got = m(obs)
        want = _exact(m, obs).detach()
        assert m._fused is not None and m._fused[1] is not None
        e = float((got.double() - want).norm() / want.norm())
        assert e < 2e-6 * (len(hidden) + 1), (act, norm, e)


def test_record_follows_the_parameters_and_falls_back(monkeypatch):
    m = _model((48,), 12, [64, 32], "elu", True)
    obs = {"g0": torch.randn(100, 48, device="cuda")}
    with torch.no_grad():
        a = m(obs)
        for p in m.parameters():  # new storage, other values
            p.data = p.data.clone() * 1.5
        b = m(obs)
        assert float((b.double() - _exact(m, obs)).norm() / b.norm()) < 1e-5 and not torch.equal(a, b)
        m.obs_normalizer._mean += 1.0  # in place
        c = m(obs)
        assert float((c.double() - _exact(m, obs)).norm() / c.norm()) < 1e-5 and not torch.equal(b, c)
        monkeypatch.setattr(models, "FUSED_ROWS", 0)
        d = m(obs)
        assert float((c - d).norm() / d.norm()) < 1e-5
    wide = _model((48,), 12, [1100, 32], "elu", False)  # a layer input past the kernel's width
    with torch.no_grad():
        y = wide(obs)
    assert wide._fused is None or wide._fused[1] is None
    assert float((y.double() - _exact(wide, obs)).norm() / y.norm()) < 1e-5


def test_rows_are_independent():
    """A NaN or an infinity in one row's observations stays in that row."""
    m = _model((48,), 12, [512, 256, 128], "elu", False)
    x = torch.randn(40, 48, device="cuda")
    with torch.no_grad():
        clean = m({"g0": x})
        x[3, 7], x[20, 0] = float("nan"), float("inf")
        y = m({"g0": x})
    assert torch.isnan(y[3]).all() and not torch.isfinite(y[20]).all()
    keep = [i for i in range(40) if i not in (3, 20)]
    assert torch.equal(y[keep], clean[keep])


@pytest.mark.parametrize("rows", [1, 16, 17, 250])
@pytest.mark.parametrize("widths,actions,hidden", [((48,), 12, [512, 256, 128]), ((33, 3), 65, [40, 70]),
                                                   ((20,), 1, [17, 1000, 30, 64, 18]), ((64,), 130, [128, 64, 66, 200])])
def test_launches_of_two_layers_give_the_one_launch_forward(monkeypatch, rows, widths, actions, hidden):
    """Three layers to six (an even and an odd count), slices of whole and of partial tiles, widths off 16 bytes: the
    same bits."""
    monkeypatch.setattr(models, "PAIR_WEIGHTS", 0)
    m = _model(widths, actions, hidden, "elu", True)
    obs = {f"g{i}": torch.randn(rows, w, device="cuda") for i, w in enumerate(widths)}
    with torch.inference_mode():
        monkeypatch.setattr(models, "PAIR_ROWS", 0)
        one = m(obs)
        monkeypatch.setattr(models, "PAIR_ROWS", 1024)
        assert m._fused[2] > 0
        assert torch.equal(m(obs), one)
