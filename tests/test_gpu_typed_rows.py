"""fp32 typed products of rows sorted by type (ga_segment_mm, _stacked, _gated): steps and blocks of
the kernel, types without rows and ragged chunks, values that are not finite, against float64."""
import numpy as np
import pytest
import torch

from graphiler_amd import ops, prepare_graph
from helpers import TOL_F32, assert_close

pytestmark = pytest.mark.gpu


def _nodes(rng, rows, types, device):
    p = rng.random(types)
    p[types // 2] = 0.0                     # a type without rows
    ntype = np.sort(rng.choice(types, rows, p=p / p.sum()))
    src = rng.integers(0, rows, 2 * rows)
    g = prepare_graph(src, src[::-1].copy(), rows, device=device, ntype_of=ntype, num_ntypes=types)
    return ntype, g


def _want(x, w, ntype):
    out = np.empty((x.shape[0], w.shape[2]))
    size = np.empty_like(out)
    with np.errstate(invalid="ignore"):
        for t in range(w.shape[0]):
            at = ntype == t
            out[at] = x[at].astype(np.float64) @ w[t]
            size[at] = np.abs(x[at]).astype(np.float64) @ np.abs(w[t])
    return out, size


@pytest.mark.parametrize("k", [4, 28, 32, 36, 64, 100, 128])
@pytest.mark.parametrize("m", [16, 32, 64, 128, 192])
@pytest.mark.parametrize("rows,types", [(1, 2), (63, 3), (65, 2), (3000, 70)])
def test_products(device, k, m, rows, types):
    rng = np.random.default_rng(k + m + rows)
    ntype, g = _nodes(rng, rows, types, device)
    x = rng.standard_normal((rows, k)).astype(np.float32)
    ws = [rng.standard_normal((types, k, m)).astype(np.float32) for _ in range(3)]
    dx, dw = torch.from_numpy(x).to(device), [torch.from_numpy(w).to(device) for w in ws]
    stacked = ops.SegmentMMNodeStacked(dx, dw, g)
    for w, d, s in zip(ws, dw, stacked):
        want, size = _want(x, w, ntype)
        got = ops.SegmentMMNode(dx, d, g)
        assert_close(got.cpu().numpy(), want, TOL_F32, "typed rows", mag=size)
        assert torch.equal(got, s)
    scale = torch.rand(rows, device=device)
    assert torch.equal(ops.SegmentMMNode(dx, dw[0], g, row_scale=scale), stacked[0] * scale[:, None])
    gate = torch.randn(types, device=device)
    want, size = _want(x, ws[0], ntype)
    for sigmoid in (True, False):
        f = (torch.sigmoid(gate.double()) if sigmoid else gate.double()).cpu().numpy()[ntype][:, None]
        got = ops.SegmentMMNodeGated(dx, dw[0], gate, g, sigmoid=sigmoid)
        assert_close(got.cpu().numpy(), want * f, TOL_F32, "gate", mag=size * np.abs(f))


@pytest.mark.parametrize("value", [np.inf, -np.inf, np.nan])
@pytest.mark.parametrize("m", [16, 64])
def test_values_that_are_not_finite(device, value, m):
    """The same rows and columns as a plain product, infinities with their signs."""
    rng = np.random.default_rng(m)
    rows, types, k = 500, 4, 64
    ntype, g = _nodes(rng, rows, types, device)
    x = rng.standard_normal((rows, k)).astype(np.float32)
    w = rng.standard_normal((types, k, m)).astype(np.float32)
    x[[3, 250], [5, 63]] = value
    w[0, 7, 2] = value
    got = ops.SegmentMMNode(torch.from_numpy(x).to(device), torch.from_numpy(w).to(device), g).cpu().numpy()
    want, _ = _want(x, w, ntype)
    fin = np.isfinite(want)
    assert np.array_equal(np.isnan(got), np.isnan(want))
    assert np.array_equal(got[~fin & ~np.isnan(want)], want[~fin & ~np.isnan(want)].astype(np.float32))
    assert np.abs(got[fin] - want[fin]).max() <= TOL_F32 * np.abs(want[fin]).max()


@pytest.mark.parametrize("k", [4, 32, 64, 128])
@pytest.mark.parametrize("m", [16, 32, 64])
def test_products_that_overflow_small_operands_and_single_products(device, k, m):
    """The range and the rounding of fp32 products: a product beyond the largest float is an infinity
    with its sign, operands of 2^-122 keep their bits, a lone product has one rounding's error (its
    pieces are added smallest first: what comes before the last addition is 2^-8 of it)."""
    rng = np.random.default_rng(k + m)
    rows, types = 700, 3
    ntype, g = _nodes(rng, rows, types, device)
    dev = lambda a: torch.from_numpy(a).to(device)
    x = rng.standard_normal((rows, k)).astype(np.float32)
    w = rng.standard_normal((types, k, m)).astype(np.float32)
    big, wide = x.copy(), w.copy()
    big[[1, 300, 699]] = 0.0                 # one product a sum that overflows, at most
    big[[1, 300, 699], [0, k - 1, k // 2]] = 3e38, -3e38, 3.3e38
    wide[:, k - 1, 3], wide[:, 0, 5] = 3e38, -3.2e38
    want, _ = _want(big, wide, ntype)
    with np.errstate(over="ignore"):
        want = want.astype(np.float32)
    got = ops.SegmentMMNode(dev(big), dev(wide), g).cpu().numpy()
    assert np.isinf(want).any() and not np.isnan(got).any()
    assert np.array_equal(got[np.isinf(want)], want[np.isinf(want)])
    assert np.isfinite(got[np.isfinite(want)]).all()
    small = x * np.float32(2.0 ** -122)
    want, size = _want(small, w, ntype)
    got = ops.SegmentMMNode(dev(small), dev(w), g).cpu().numpy().astype(np.float64)
    assert (np.abs(got - want) <= (k + 8) * 2.0 ** -24 * size + k * 2.0 ** -149).all()
    lone = np.zeros_like(x)
    at = rng.integers(0, k, rows)
    lone[np.arange(rows), at] = x[:, 0]
    got = ops.SegmentMMNode(dev(lone), dev(w), g).cpu().numpy()
    want = x[:, :1].astype(np.float64) * w[ntype, at]
    assert (np.abs(got - want) <= (1 + 2.0 ** -6) * 2.0 ** -24 * np.abs(want)).all()
