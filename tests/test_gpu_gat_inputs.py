"""The GAT layer over its inputs (ops.gat_inputs, ga_gat_inputs) against the layer in float64: heads
and widths, rows longer than a piece, rows without edges, inputs that are not finite."""
import numpy as np
import pytest
import torch

from graphiler_amd import layers, ops, prepare_graph
from helpers import TOL_BF16, assert_close

pytestmark = pytest.mark.gpu


def _graph(rng, n, e, device, hub=0):
    src, dst = rng.integers(0, n, e), (n * rng.random(e) ** 2).astype(np.int64)
    dst[:hub] = n // 3
    dst[dst == n - 1] = 0               # the last node has no in-edges
    return src, dst, prepare_graph(src, dst, n, device=device)


def _reference(src, dst, n, x, w, a, slope, act):
    heads, dim = a.shape[1:]
    z = (x.double() @ w.double()).view(n, heads, dim)
    el, er = (z * a[0].double()).sum(2), (z * a[1].double()).sum(2)
    s, d = torch.from_numpy(src).to(x.device), torch.from_numpy(dst).to(x.device)
    score = torch.nn.functional.leaky_relu(el[s] + er[d], slope)
    top = torch.full((n, heads), -np.inf, dtype=torch.float64, device=x.device)
    top = top.scatter_reduce(0, d[:, None].expand_as(score), score, "amax")
    p = torch.exp(score - top[d])
    p = p / torch.zeros_like(top).index_add_(0, d, p)[d]
    out = torch.zeros(n, heads, dim, dtype=torch.float64, device=x.device).index_add_(0, d, z[s] * p[:, :, None])
    out = out.view(n, -1)
    return torch.relu(out) if act == "relu" else torch.nn.functional.elu(out) if act == "elu" else out


@pytest.mark.parametrize("heads,dim", [(1, 16), (1, 64), (2, 32), (2, 128), (4, 16), (4, 64), (4, 192), (8, 32), (8, 64)])
@pytest.mark.parametrize("k", [1, 8, 31, 56, 62, 100, 112])
def test_against_float64(device, heads, dim, k):
    """k: one to four steps of the product, rows of one and of two lines, loads of 2 to 16 bytes.
    A row of 900 in-edges is walked in pieces (256 slots for this many edges)."""
    rng = np.random.default_rng(heads * dim + k)
    n, e = 1003, 9000
    src, dst, g = _graph(rng, n, e, device, hub=900)
    assert g.rows_by_length().n_light < n
    gen = torch.Generator(device=device).manual_seed(k)
    x = torch.randn(n, k, device=device, generator=gen).bfloat16()
    w = (torch.randn(k, heads * dim, device=device, generator=gen) / k ** 0.5).bfloat16()
    a = torch.randn(2, heads, dim, device=device, generator=gen) / dim ** 0.5
    for act in (None, "relu", "elu"):
        got = ops.gat_inputs(x, w, a[0], a[1], g, 0.2, act)
        want = _reference(src, dst, n, x, w, a, 0.2, act)
        # rounding the result is all that bf16 costs here: 2^-9 of a value
        assert ((got.double() - want).abs() <= 2 ** -8 * want.abs() + 1e-5 * want.abs().max()).all()
        assert not got[n - 1].any()
        assert torch.equal(got.view(torch.int16), ops.gat_inputs(x, w, a[0], a[1], g, 0.2, act).view(torch.int16))


@pytest.mark.parametrize("n,e", [(1, 1), (15, 40), (16, 3000), (17, 17), (5000, 3), (40, 20000)])
def test_graph_sizes(device, n, e):
    rng = np.random.default_rng(n + e)
    src, dst = rng.integers(0, n, e), rng.integers(0, n, e)
    g = prepare_graph(src, dst, n, device=device)
    x = torch.randn(n, 60, device=device).bfloat16()
    w = (torch.randn(60, 256, device=device) / 8).bfloat16()
    a = torch.randn(2, 4, 64, device=device) / 8
    got, want = ops.gat_inputs(x, w, a[0], a[1], g, 0.2), _reference(src, dst, n, x, w, a, 0.2, None)
    assert_close(got.double().cpu().numpy(), want.cpu().numpy(), TOL_BF16, "layer over its inputs")


@pytest.mark.parametrize("value", [float("inf"), float("-inf"), float("nan")])
@pytest.mark.parametrize("heads,dim", [(1, 64), (4, 64), (8, 32)])
def test_inputs_that_are_not_finite_stay_with_their_rows(device, value, heads, dim):
    rng = np.random.default_rng(heads)
    n, e, k = 800, 9000, 100
    src, dst, g = _graph(rng, n, e, device, hub=700)
    x = torch.randn(n, k, device=device).bfloat16()
    w = (torch.randn(k, heads * dim, device=device) / k ** 0.5).bfloat16()
    a = torch.randn(2, heads, dim, device=device) / dim ** 0.5
    want = _reference(src, dst, n, x, w, a, 0.2, None)
    bad = [0, 5, int(src[0])]           # row 0 is also what lanes without a slot read
    x[bad, 99] = value
    got = ops.gat_inputs(x, w, a[0], a[1], g, 0.2).double()
    touched = np.zeros(n, dtype=bool)
    touched[dst[np.isin(src, bad)]] = True
    touched[bad] = True                 # their own terms as destinations
    clean = torch.from_numpy(~touched).to(device)
    assert clean.any() and torch.isfinite(got[clean]).all()
    assert ((got - want)[clean].abs() <= 2 ** -8 * want[clean].abs() + 1e-5 * want.abs().max()).all()
    hit = np.zeros(n, dtype=bool)
    hit[dst[np.isin(src, bad)]] = True
    assert hit[n // 3] and np.bincount(dst, minlength=n)[n // 3] > 256     # a row in pieces is among them
    assert not torch.isfinite(got[torch.from_numpy(hit).to(device)]).any()


@pytest.mark.parametrize("value", [float("inf"), float("-inf"), float("nan")])
@pytest.mark.parametrize("heads,dim", [(1, 16), (2, 32), (4, 64), (8, 64)])
def test_weights_that_are_not_finite(device, value, heads, dim):
    """A value of W that is not finite makes its head's logits so, and with them that head of every
    destination that has in-edges; one without stays a row of zeros, and so do the other heads."""
    rng = np.random.default_rng(heads + dim)
    n, e, k = 500, 1200, 60             # a tenth of the nodes have no in-edges
    src, dst, g = _graph(rng, n, e, device, hub=400)
    x = torch.randn(n, k, device=device).bfloat16()
    w = (torch.randn(k, heads * dim, device=device) / k ** 0.5).bfloat16()
    a = torch.randn(2, heads, dim, device=device) / dim ** 0.5
    want = _reference(src, dst, n, x, w, a, 0.2, "elu")
    w[3, dim // 2] = value
    got = ops.gat_inputs(x, w, a[0], a[1], g, 0.2, "elu").double()
    fed = torch.zeros(n, dtype=torch.bool, device=device)
    fed[torch.from_numpy(dst).to(device)] = True
    assert (~fed).sum() > 16 and (got[~fed] == 0).all()
    assert not torch.isfinite(got[fed, :dim]).any()
    near = (got - want)[:, dim:].abs() <= 2 ** -8 * want[:, dim:].abs() + 1e-5 * want.abs().max()
    assert near.all()


def test_the_layer_takes_it_and_falls_back(device, monkeypatch):
    rng = np.random.default_rng(5)
    n, e, k = 3000, 600_000, 50
    src, dst, g = _graph(rng, n, e, device)
    x = torch.randn(n, k, device=device).bfloat16()
    w = (torch.randn(k, 512, device=device) / k ** 0.5).bfloat16()
    a = torch.randn(2, 8, 64, device=device) / 8
    assert ops.gat_inputs_preferred(k, 8, 512, g.num_edges)
    want = ops.gat_inputs(x, w, a[0].contiguous(), a[1].contiguous(), g, 0.2, "elu")
    assert torch.equal(layers.gat_layer(g, x, w, a, 8, 0.2, activation="elu"), want)
    plain = layers.gat_layer(g, x, w, a, 8, 0.2, fused=False, activation="elu")
    assert_close(want.float().cpu().numpy(), plain.float().cpu().numpy(), 2 * TOL_BF16, "against the operators")
    for kk, heads, dim in ((125, 4, 64), (50, 3, 64), (50, 4, 48)):
        xx, ww = torch.randn(n, kk, device=device).bfloat16(), torch.randn(kk, heads * dim, device=device).bfloat16()
        aa = torch.randn(heads, dim, device=device)
        assert ops.gat_inputs(xx, ww, aa, aa, g) is None
    # a graph whose order of rows is not there is not given one inside a capture
    fresh = prepare_graph(src, dst, n, device=device)
    layers.gat_layer(g, x, w, a, 8, 0.2)
    fresh.in_row_of_slot, fresh.workspace(64 << 20)
    monkeypatch.setattr(torch.cuda, "is_current_stream_capturing", lambda: True)
    assert ops.gat_inputs(x, w, a[0].contiguous(), a[1].contiguous(), fresh) is None
    assert "rows_by_length" not in fresh._cache
