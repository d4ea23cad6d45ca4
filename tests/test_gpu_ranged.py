"""The GEMMs with known operand ranges (fp16x3, csrc/gemm_f16.hpp) and the largest-magnitude slots behind them.

Tolerances: fp16x3 leaves at most 2^-22 of each |a||b| product (2 x 2^-23 from the operands' residuals, and lo.lo), i.e.
2.4e-7 of the |A||B| bound, plus fp32 accumulation; the bars are the fp32 GEMMs' own (2e-6 of the result's norm and of
each element's bound), and the error must be no larger than the plain kernels' on the same problem (plus 2e-8: at k = 64
both are near the rounding of one product).  Launches with a k below 64 run the plain kernels: the same bits."""

from __future__ import annotations

import pytest
import torch

from tt_rsl_rl_amd import _lib as L
from tt_rsl_rl_amd import ops

pytestmark = pytest.mark.gpu


def _buf(rows, cols, scale=1.0, seed=0):
    """[rows, cols] view of rows padded to whole 16 bytes, the padding poisoned."""
    g = torch.Generator("cuda").manual_seed(seed)
    t = torch.full((rows, -(-cols // 4) * 4), float("nan"), device="cuda")
    t[:, :cols] = torch.randn(rows, cols, device="cuda", generator=g) * scale
    return t[:, :cols]


def _slots(*tensors):
    s = ops.new_amax(len(tensors), "cuda")
    ops.amax([(t, s[i]) for i, t in enumerate(tensors)])
    return list(s)


def _largest(slots) -> float:
    return float(slots.view(torch.float32).max())


def _check(got, base, want, bound, k):
    e = float((got.double() - want).norm() / want.norm())
    e0 = float((base.double() - want).norm() / want.norm())
    assert e < 2e-6 and float(((got.double() - want).abs() / bound.clamp(min=1e-300)).max()) < 2e-6
    if k < 64:
        assert torch.equal(got, base)
    else:
        assert not torch.equal(got, base), "the same kernel ran"
        assert e <= e0 + 2e-8, (e, e0)


def test_amax_slots():
    x = _buf(1000, 37, seed=1)
    x[3, 5], x[700, 36] = -9.5, float("inf")
    w = torch.randn(77, 13, device="cuda")
    z = torch.zeros(50, 8, device="cuda")
    clear = torch.full((3, L.AMAX_WORDS), 5, dtype=torch.int32, device="cuda")
    s = ops.new_amax(4, "cuda")
    s.fill_(0x7f000000)  # (stale contents are replaced)
    s[:, 1:32] = 0
    s = s * (torch.arange(L.AMAX_WORDS, device="cuda") % 32 == 0)
    s = s.to(torch.int32)
    ops.amax([(x, s[0]), (w, s[1]), (z, s[2]), (z, s[3], 2.0)], clear)
    finite = x[torch.isfinite(x)]
    assert _largest(s[0]) == float(finite.abs().max())
    assert _largest(s[1]) == float(w.abs().max())
    assert _largest(s[2]) == 0.0 and _largest(s[3]) == 2.0
    assert int(clear.abs().max()) == 0


# tile edges (128 rows, 64 / 128 columns, 32-deep slabs with 16-deep halves), remainders, one and many tiles
@pytest.mark.parametrize("rows,k,n", [(1, 4, 4), (127, 16, 64), (128, 17, 68), (129, 31, 128), (130, 32, 132),
                                      (300, 33, 60), (257, 48, 512), (300, 64, 60), (257, 65, 512), (513, 100, 200), (4096, 37, 100),
                                      (33000, 99, 256), (20000, 240, 512), (40001, 512, 256)])
@pytest.mark.parametrize("act", ["elu", "tanh", "relu", "gelu"])
def test_forward(rows, k, n, act):
    x, w = _buf(rows, k, 3.0, 1), _buf(n, -(-k // 4) * 4, 0.1, 2).contiguous()
    if k % 4:  # (a weight with padded rows, its padding zero, against an input block read as wide)
        w[:, k:] = 0.0
        xw = torch.cat([x, torch.full((rows, w.shape[1] - k), 2.5, device="cuda")], 1)
    else:
        xw = x
    b = torch.randn(n, device="cuda")
    code = L.ACTIVATIONS[act]
    h, h0 = _buf(rows, n), _buf(rows, n)
    sx, sw = _slots(xw, w)
    out = ops.new_amax(1, "cuda")[0]
    ops.linear_fwd([(xw, w, b, None, h)], rows, act=code, ranges=[(sx, sw, out)])
    ops.linear_fwd([(xw, w, b, None, h0)], rows, act=code)
    z = x.double() @ w[:, :k].double().t() + b.double()
    f = {"elu": torch.nn.functional.elu, "tanh": torch.tanh, "relu": torch.relu, "gelu": torch.nn.functional.gelu}[act]
    want = f(z)
    assert _largest(out) == float(h.abs().max())
    # (every one of these activations has a slope of at most 1.13)
    bound = 1.13 * (x.double().abs() @ w[:, :k].double().abs().t() + b.double().abs()) + want.abs()
    _check(h, h0, want, bound, k)


@pytest.mark.parametrize("rows,k,n", [(1, 4, 4), (127, 17, 64), (129, 31, 68), (300, 33, 132), (513, 100, 200), (129, 64, 4), (127, 81, 68),
                                      (4096, 37, 100), (33000, 256, 512), (40001, 128, 48)])
@pytest.mark.parametrize("act", ["elu", "tanh", "relu", None])
def test_input_grad(rows, k, n, act):
    dz, w = _buf(rows, k, 1e-6, 1), _buf(k, n, 0.1, 2).contiguous()
    src = _buf(rows, n, 0.4, 3)
    d, d0 = _buf(rows, n), _buf(rows, n)
    sd, sw = _slots(dz, w)
    out = ops.new_amax(1, "cuda")[0]
    ws = ops.Workspace("cuda")
    code = L.ACTIVATIONS[act] if act else L.PPO_ACT_ELU
    for dst, rng in ((d, [(sd, sw, out)]), (d0, None)):
        ops.linear_bwd_dx([(dz, w, src if act else None, dst)], rows, ws, elu_from_output=True, act=code, ranges=rng)
    s = src.double()
    slope = {"elu": torch.where(s > 0, 1.0, s + 1), "tanh": 1 - s * s, "relu": (s > 0).double(), None: torch.ones_like(s)}[act]
    want = (dz.double() @ w.double()) * slope
    assert _largest(out) == float(d.abs().max())
    _check(d, d0, want, (dz.double().abs() @ w.double().abs()) * slope.abs() + 1e-30, k)


@pytest.mark.parametrize("rows", [1, 63, 64, 65, 95, 96, 97, 1003, 3006, 40001])
def test_weight_grad(rows):
    """Grouped problems, narrow (128 x 64 tiles) and wide, one column to several tiles; below 64 rows the plain kernels
    run.  The bias sums stay the fp64 ones."""
    shapes = [(64, 48), (29, 128), (1, 100), (132, 200), (256, 60)]
    probs, base, rng, want = [], [], [], []
    for i, (o, k) in enumerate(shapes):
        dz, x = _buf(rows, o, 1e-6, 10 + i), _buf(rows, k, 2.0, 20 + i)
        sd, sx = _slots(dz, x)
        dw, db = torch.empty(o, k, device="cuda"), torch.empty(o, device="cuda")
        probs.append((dz, x, dw, db))
        base.append((dz, x, torch.empty_like(dw), torch.empty_like(db)))
        rng.append((sd, sx, None))
        want.append((dz.double().t() @ x.double(), dz.double().abs().t() @ x.double().abs(), dz.double().sum(0)))
    ops.linear_bwd_dw(probs, rows, ranges=rng)
    ops.linear_bwd_dw(base, rows)
    for (_, _, dw, db), (_, _, dw0, db0), (w64, bound, b64) in zip(probs, base, want):
        _check(dw, dw0, w64, bound, rows)
        assert torch.allclose(db.double(), b64, rtol=1e-6, atol=1e-12)


def test_zero_tiny_and_non_finite_operands():
    """All-zero operands give zeros; an operand of subnormal magnitude keeps finite results; a NaN or an infinity stays
    in the rows it belongs to."""
    rows, k, n = 200, 64, 128
    b = torch.zeros(n, device="cuda")
    for scale in (0.0, 1e-40, 1e30):
        x, w = _buf(rows, k, 1.0, 1) * scale, _buf(n, k, 0.1, 2).contiguous()
        z = torch.empty(rows, n, device="cuda")
        sx, sw = _slots(x, w)
        ops.linear_fwd([(x, w, b, z, None)], rows, act=0, ranges=[(sx, sw, None)])
        want = x.double() @ w.double().t()
        assert torch.isfinite(z).all()
        assert float((z.double() - want).norm()) <= 2e-6 * float(want.norm()) + 1.4e-45 * z.numel() ** 0.5
    x = _buf(rows, k, 1.0, 1)
    x[7, 3], x[90, 60] = float("nan"), float("inf")
    sx, sw = _slots(x, w)
    ops.linear_fwd([(x, w, b, z, None)], rows, act=0, ranges=[(sx, sw, None)])
    bad = torch.zeros(rows, dtype=torch.bool, device="cuda")
    bad[[7, 90]] = True
    assert not torch.isfinite(z[bad]).any()
    want = x[~bad].double() @ w.double().t()
    assert float((z[~bad].double() - want).norm() / want.norm()) < 2e-6


def _rel(got, want) -> float:
    return float((got.double() - want).norm() / want.norm())


# (of whom, what): one element, a whole row, a column of another unit in the activations; a row or column of the weights
_SPREADS = [("x", "element", -1e10), ("x", "element", 1e15), ("x", "element", -1e20), ("x", "element", 3e38), ("x", "row", 1e12),
            ("x", "rows", 1e20), ("x", "column", 1e-11), ("x", "column", 1e9), ("w", "row", 1e-10), ("w", "row", 1e12),
            ("w", "column", 1e-12), ("x", "none", 1.0)]


@pytest.mark.parametrize("whose,what,size", _SPREADS)
def test_operands_of_wide_range_keep_their_small_parts(whose, what, size):
    """What lies far below the tensor's largest magnitude keeps its digits: every other row of a forward, every row and
    column of a weight-grad, as in the plain kernels.  (fp16x3 scales a tensor by its largest magnitude.)"""
    rows, k, n = 1000, 96, 200
    x, w = _buf(rows, k, 1.0, 1).clone(), _buf(n, k, 0.1, 2).clone()
    dz = _buf(rows, n, 1e-4, 3).clone()
    t = x if whose == "x" else w
    odd_rows = torch.zeros(rows, dtype=torch.bool, device="cuda")
    if what == "element":
        t[7, 5], odd_rows[7] = size, True
    elif what == "row":
        t[7] *= size
        odd_rows[7] = whose == "x"
    elif what == "rows":  # a sentinel in every 16th row, all of its columns
        odd_rows[::16] = True
        t[odd_rows] = size
    elif what == "column":
        t[:, 5] *= size
    dz[odd_rows] = 0.0  # (a saturated unit's: the row is in no sum)
    b = torch.randn(n, device="cuda") * (0.0 if whose == "w" else 1.0)
    z, z0 = torch.empty(rows, n, device="cuda"), torch.empty(rows, n, device="cuda")
    sx, sw, sd = _slots(x, w, dz)
    ops.linear_fwd([(x, w, b, z, None)], rows, act=0, ranges=[(sx, sw, None)])
    ops.linear_fwd([(x, w, b, z0, None)], rows, act=0)
    want = x.double() @ w.double().t() + b.double()
    ok = ~odd_rows
    for i in ([slice(None)] if whose == "x" else [7, slice(0, 7)]):  # (each output unit by itself: its weights' scale)
        e, e0 = _rel(z[ok][:, i], want[ok][:, i]), _rel(z0[ok][:, i], want[ok][:, i])
        assert e < 1e-6 and e <= e0 + 5e-8, (i, e, e0)

    dw, dw0, db = torch.empty(n, k, device="cuda"), torch.empty(n, k, device="cuda"), torch.empty(n, device="cuda")
    ops.linear_bwd_dw([(dz, x, dw, db)], rows, ranges=[(sd, sx, None)])
    ops.linear_bwd_dw([(dz, x, dw0, db)], rows)
    want = dz.double().t() @ x.double()
    for c in (5, 6):  # (each column by itself: an optimiser rescales it)
        e, e0 = _rel(dw[:, c], want[:, c]), _rel(dw0[:, c], want[:, c])
        assert e < 1e-6 and e <= 1.5 * e0 + 5e-8, (c, e, e0)

    src = torch.rand(rows, k, device="cuda")
    d, d0 = torch.empty(rows, k, device="cuda"), torch.empty(rows, k, device="cuda")
    for dst, rng in ((d, [(sd, sw, None)]), (d0, None)):
        ops.linear_bwd_dx([(dz, w, src, dst)], rows, elu_from_output=True, act=L.PPO_ACT_ELU, ranges=rng)
    want = dz.double() @ w.double()
    for c in (5, 6):
        e, e0 = _rel(d[:, c], want[:, c]), _rel(d0[:, c], want[:, c])
        assert e < 1e-6 and e <= e0 + 5e-8, (c, e, e0)


def test_a_wide_problem_leaves_the_others_of_its_launch():
    """Two problems per launch, one with an outlier: the other one's bits are those of its launch alone."""
    rows, k, n = 700, 64, 132
    x, w, b = _buf(rows, k, 1.0, 1).clone(), _buf(n, k, 0.1, 2).clone(), torch.randn(n, device="cuda")
    far = x.clone()
    far[3, 3] = 1e15
    dz = _buf(rows, n, 1e-4, 3).clone()
    sx, sf, sw, sd = _slots(x, far, w, dz)
    h = [torch.empty(rows, n, device="cuda") for _ in range(3)]
    out = ops.new_amax(3, "cuda")
    ops.linear_fwd([(x, w, b, None, h[0])], rows, act=L.PPO_ACT_ELU, ranges=[(sx, sw, out[0])])
    ops.linear_fwd([(far, w, b, None, h[1]), (x, w, b, None, h[2])], rows, act=L.PPO_ACT_ELU,
                   ranges=[(sf, sw, out[1]), (sx, sw, out[2])])
    assert torch.equal(h[2], h[0]) and _largest(out[2]) == _largest(out[0])
    keep = torch.arange(rows, device="cuda") != 3
    assert _rel(h[1][keep], h[0][keep].double()) < 1e-6
    assert _largest(out[1]) == float(h[1].abs().max())
    g = [torch.empty(n, k, device="cuda") for _ in range(3)]
    db = torch.empty(n, device="cuda")
    ops.linear_bwd_dw([(dz, far, g[1], db), (dz, x, g[2], db)], rows, ranges=[(sd, sf, None), (sd, sx, None)])
    ops.linear_bwd_dw([(dz, x, g[0], db), (dz, x, g[0], db)], rows, ranges=[(sd, sx, None), (sd, sx, None)])
    assert torch.equal(g[2], g[0])


@pytest.mark.parametrize("k", [48, 64])  # (below 64 a layer runs the plain kernels, and tracks its output in those)
@pytest.mark.parametrize("n", [128, 120])
@pytest.mark.parametrize("value,every", [(1e25, 500), (3e38, 500), (1e25, 16), (1e12, 4)])
def test_outliers_that_a_layer_writes(k, n, value, every):
    """The range that a forward leaves of its output carries outliers and infinities to the next layers' launches, also
    where each part holds one (every 16th row): the other rows keep their values."""
    rows = 1000
    x, w1, w2 = _buf(rows, k, 1.0, 1).clone(), _buf(n, k, 0.1, 2).clone(), _buf(n, n, 0.1, 3).clone()
    b = torch.zeros(n, device="cuda")
    odd = torch.arange(rows, device="cuda") % every == 11 % every
    x[odd] = value
    w1[:, 0] = w1[:, 0].abs() * 10
    h1, h2, z = (torch.empty(rows, n, device="cuda") for _ in range(3))
    out = ops.new_amax(3, "cuda")
    sx, sw1, sw2 = _slots(x, w1, w2)
    ops.linear_fwd([(x, w1, b, None, h1)], rows, act=L.PPO_ACT_ELU, ranges=[(sx, sw1, out[0])])
    ops.linear_fwd([(h1, w2, b, None, h2)], rows, act=L.PPO_ACT_ELU, ranges=[(out[0], sw2, out[1])])
    ops.linear_fwd([(h2, w2, b, z, None)], rows, act=0, ranges=[(out[1], sw2, None)])
    elu = torch.nn.functional.elu
    want = elu(elu(x[~odd].double() @ w1.double().t()) @ w2.double().t()) @ w2.double().t()
    assert _rel(z[~odd], want) < 1e-6
    # the gradient of a weight whose rows with outliers are zero in dz, and dz's own way down
    dz = _buf(rows, n, 1e-4, 4).clone()
    dz[odd] = 0.0
    (sd,), src = _slots(dz), torch.rand(rows, n, device="cuda")
    dw, db = torch.empty(n, n, device="cuda"), torch.empty(n, device="cuda")
    ops.linear_bwd_dw([(dz, h1, dw, db)], rows, ranges=[(sd, out[0], None)])
    if value < 1e30:  # (0 x infinity)
        assert _rel(dw, dz[~odd].double().t() @ elu(x[~odd].double() @ w1.double().t())) < 1e-6
    dz[odd] = 1e15
    (sd,) = _slots(dz)
    d1, d0 = torch.empty(rows, n, device="cuda"), torch.empty(rows, n, device="cuda")
    for a, c, s, o in ((dz, d1, sd, out[2]), (d1, d0, out[2], None)):
        ops.linear_bwd_dx([(a, w2, src, c)], rows, elu_from_output=True, act=L.PPO_ACT_ELU, ranges=[(s, sw2, o)])
    assert _rel(d0[~odd], dz[~odd].double() @ w2.double() @ w2.double()) < 1e-6


def _smallest(slots) -> float:
    """The largest magnitude of the smallest part that the slots know of (csrc/amax.hpp)."""
    low = (slots.view(-1, 32)[:, 1].to(torch.int64) & 0xffffffff).max()
    return float((0x7f800000 - (low & 0x7fffffff)).to(torch.int32).view(torch.float32))


def test_ranges_of_many_rows_raised_in_pieces():
    """Raising by one block of rows after another (more blocks than slots) finds what one pass finds, the smallest part as
    well (here one row, or where that is zero one column): any widths, off 16 bytes, padding left out."""
    for rows, cols in ((5000, 240), (70001, 3), (333, 700), (1000, 65)):
        x = _buf(rows, cols, 1.0, 5)
        x[17] *= 1e-9
        part = min(float(x[17, c:c + 256].abs().max()) for c in range(0, cols, 256))
        a, b = ops.new_amax(2, "cuda")
        for _ in range(2):
            ops.amax([(x, a)])
            b.zero_()
            for piece in (x[:rows // 3], x[rows // 3:]):
                ops.amax([(piece, b)], raising=True)
            assert _largest(a) == _largest(b) == float(x.abs().max())
            assert _smallest(a) == part and _smallest(b) <= part
            x[17] = 0.0  # (a part of zeros is none)
            x[:, 2] *= 1e-12
            part = float("inf")
            for r0 in range(0, rows, max(16, -(-rows // 64))):
                part = min(part, float(x[r0:r0 + max(16, -(-rows // 64)), 2].abs().max()))
        ops.amax([(x[17:18], a)])
        assert _largest(a) == 0.0 and int(a.abs().max()) == 0
        x = _buf(rows, cols, 1.0, 5)
        x[17] *= 1e-9
        ops.amax([(x, a)], coarse=True)
        assert _smallest(a) > 1e-4


@pytest.mark.parametrize("activation,every,actions", [("tanh", 256, 8), ("elu", 256, 8), ("tanh", 8, 8), ("tanh", 8, 37)])
def test_update_with_a_sentinel_observation(activation, every, actions, monkeypatch):
    """One element of a row at -1e20 (a sensor's sentinel), in one row or in every eighth, in an update large enough for
    fp16x3: the parameters are those of the plain kernels' update."""
    from types import SimpleNamespace

    from tt_rsl_rl_amd import engine
    from tt_rsl_rl_amd.ppo import PPO

    n, steps = 256, 4

    def run(ranged):
        monkeypatch.setattr(engine, "RANGED_ROWS", 1 if ranged else 1 << 40)
        torch.manual_seed(0)
        model = dict(class_name="MLPModel", hidden_dims=[128, 64], activation=activation)
        cfg = dict(algorithm=dict(class_name="tt_rsl_rl_amd.ppo:PPO", num_learning_epochs=1, num_mini_batches=1,
                                  schedule="fixed", optimizer="sgd", learning_rate=1.0),
                   actor=dict(model, distribution_cfg=dict(class_name="GaussianDistribution")), critic=model,
                   obs_groups={"actor": ["g"], "critic": ["g"]}, num_steps_per_env=steps)
        alg = PPO.construct_algorithm({"g": torch.zeros(n, 96)}, SimpleNamespace(num_envs=n, num_actions=actions), cfg, "cuda:0")
        g = torch.Generator("cuda").manual_seed(1)
        with torch.inference_mode():
            for t in range(steps):
                obs = torch.randn(n, 96, generator=g, device="cuda")
                if t == 2:
                    obs[5::every, 3] = -1e20
                alg.act({"g": obs})
                if t == 2:  # (the row's own value and action as of another policy: finite, and its ratio clipped or zero)
                    alg.transition.values[5::every] = 0.0
                    alg.transition.actions_log_prob[5::every] = 0.0
                alg.process_env_step({"g": obs}, torch.randn(n, generator=g, device="cuda"), torch.zeros(n, device="cuda"), {})
            alg.compute_returns({"g": torch.randn(n, 96, generator=g, device="cuda")})
        torch.manual_seed(2)
        before = [p.detach().clone() for m in (alg.actor, alg.critic) for p in m.parameters()]
        alg.update()
        assert alg._engine.ranged is ranged
        return [p.detach() - q for p, q in zip([p for m in (alg.actor, alg.critic) for p in m.parameters()], before)]

    for a, b in zip(run(True), run(False), strict=True):
        assert torch.equal(torch.isfinite(a), torch.isfinite(b))
        if float(b.norm()) > 0:
            assert float((a - b).norm() / b.norm()) < 1e-4


def test_an_engine_that_uses_no_ranges_allocates_none():
    """Small and recurrent updates run without slots; an engine made with mixed precision has them for when that is off."""
    from types import SimpleNamespace

    from tt_rsl_rl_amd import engine
    from tt_rsl_rl_amd.ppo import PPO

    def made(n, mixed=False, **model):
        model = dict(dict(class_name="MLPModel", hidden_dims=[16], activation="elu"), **model)
        cfg = dict(algorithm=dict(class_name="tt_rsl_rl_amd.ppo:PPO", num_mini_batches=1, use_mixed_precision=mixed),
                   actor=dict(model, distribution_cfg=dict(class_name="GaussianDistribution")), critic=model,
                   obs_groups={"actor": ["g"], "critic": ["g"]}, num_steps_per_env=2)
        alg = PPO.construct_algorithm({"g": torch.zeros(n, 4)}, SimpleNamespace(num_envs=n, num_actions=2), cfg, "cuda:0")
        alg.storage.distribution_params = ()
        return alg._get_engine()

    lstm = dict(class_name="RNNModel", rnn_type="lstm", rnn_hidden_dim=16, rnn_num_layers=1)
    n = engine.RANGED_ROWS // 2
    for e, slots in ((made(100), False), (made(n, **lstm), False), (made(n), True), (made(n, mixed=True), True)):
        assert hasattr(e, "w_max") is slots
        assert not e.ranged or slots


@pytest.mark.parametrize("act", ["tanh", "elu"])
def test_activations_are_as_close_as_the_plain_kernels(act):
    """The ranged forward's activations on exact inputs (an identity weight, 20-bit inputs that two fp16 parts hold) against
    fp64, in units of the last place: at most 1.4, and in root mean square the plain kernels' (tanhf; the longer ELU) plus
    2 % (ELU's shorter polynomial is 2e-8 off, a third of a rounding)."""
    rows, k = 1 << 15, 64
    g = torch.Generator("cuda").manual_seed(0)
    w, b, f = torch.eye(k, device="cuda"), torch.zeros(k, device="cuda"), {"tanh": torch.tanh, "elu": torch.nn.functional.elu}[act]
    worst, sq = [0.0, 0.0], [0.0, 0.0]
    for lo, hi in ((1e-3, 0.01), (0.01, 0.5), (0.5, 0.6), (0.6, 0.7), (0.69, 0.71), (0.7, 1.0), (0.99, 1.01), (1.0, 2.0), (2.0, 12.0)):
        for sign in (1.0, -1.0):
            x = torch.rand(rows, k, generator=g, device="cuda") * (hi - lo) + lo
            x = (x.view(torch.int32) & ~0xF).view(torch.float32) * sign
            sx, sw = _slots(x, w)
            want = f(x.double())
            ulp = torch.pow(2.0, torch.frexp(want.abs())[1].double() - 24)
            for i, rng in enumerate(([(sx, sw, None)], None)):
                z, h = torch.empty(rows, k, device="cuda"), torch.empty(rows, k, device="cuda")
                ops.linear_fwd([(x, w, b, z, h)], rows, act=L.ACTIVATIONS[act], ranges=rng)
                assert torch.equal(z, x)
                e = (h.double() - want).abs() / ulp
                worst[i], sq[i] = max(worst[i], float(e.max())), sq[i] + float((e ** 2).mean())
    print(act, worst, [(s / 18) ** 0.5 for s in sq])
    assert worst[0] <= 1.4 and sq[0] ** 0.5 <= 1.02 * sq[1] ** 0.5
