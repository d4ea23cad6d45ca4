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
