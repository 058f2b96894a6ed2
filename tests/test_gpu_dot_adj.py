"""Dot products over the adjacency (ga_sddmm_u_dot_v_adj) against float64: eight slots to a
lane group, rows that fill it or not, edge ids in slot order or not, rows without edges."""
import numpy as np
import pytest
import torch

from graphiler_amd import capi, ops, prepare_graph, torch_boundary

pytestmark = pytest.mark.gpu


def _graph(n, e, by_dst, seed):
    rng = np.random.default_rng(seed)
    src, dst = rng.integers(0, n, e), rng.integers(0, n, e)
    dst[: e // 3] = n - 1
    if by_dst:
        order = np.argsort(dst, kind="stable")
        src, dst = src[order], dst[order]
    return prepare_graph(src, dst, n, device="cuda:0")


def _exact(g, u, v):
    a, b = u.double()[g.COO_src], v.double()[g.COO_dst]
    return (a * b).sum(2), (a * b).abs().sum(2)


@pytest.mark.parametrize("n,e", [(1, 1), (4, 7), (9, 8), (50, 9), (300, 2049), (5000, 40_003)])
@pytest.mark.parametrize("by_dst", [False, True])
@pytest.mark.parametrize("heads,dim,bf16", [(4, 16, False), (8, 8, False), (5, 4, False), (1, 64, False),
                                            (3, 32, False), (4, 64, False), (1, 64, True), (6, 8, True),
                                            (4, 128, True)])
def test_against_float64(device, n, e, by_dst, heads, dim, bf16):
    g = _graph(n, e, by_dst, e + heads)
    gen = torch.Generator(device=device).manual_seed(dim)
    dt, code = (torch.bfloat16, capi.GA_BF16) if bf16 else (torch.float32, capi.GA_F32)
    u, v = (torch.randn(n, heads, dim, generator=gen, device=device).to(dt) for _ in range(2))
    out = torch.full((e, heads), float("nan"), device=device)
    capi.check(capi.load().ga_sddmm_u_dot_v_adj(
        g.in_row_of_slot.data_ptr(), g.in_node_indices.data_ptr(),
        None if g.in_eid_is_identity else g.in_edge_indices.data_ptr(), u.data_ptr(), v.data_ptr(),
        out.data_ptr(), e, heads, dim, code, 0), "dot")
    ref, size = _exact(g, u, v)
    # every product and addition of a head rounds to 2^-24 of at most the sum of magnitudes
    assert bool(((out.double() - ref).abs() <= size * (dim * 2.0 ** -24)).all())


def test_refused_shapes(device):
    g = _graph(20, 64, False, 1)
    lib = capi.load()
    x = torch.zeros(20 * 512 + 4, device=device)
    out = torch.empty(64 * 64, device=device)
    call = lambda u, heads, dim: lib.ga_sddmm_u_dot_v_adj(
        g.in_row_of_slot.data_ptr(), g.in_node_indices.data_ptr(), g.in_edge_indices.data_ptr(),
        u.data_ptr(), x.data_ptr(), out.data_ptr(), 64, heads, dim, capi.GA_F32, 0)
    for heads, dim in ((4, 4), (2, 12), (3, 17), (1, 128), (5, 64)):
        assert call(x, heads, dim) == capi.GA_EUNSUPPORTED
    assert call(x[1:], 4, 16) == capi.GA_EUNSUPPORTED


@pytest.mark.parametrize("e", [(1 << 15) - 1, 1 << 15])
def test_operators(device, e):
    torch_boundary.load()
    g = _graph(3000, e, False, e)
    gen = torch.Generator(device=device).manual_seed(e)
    u, v = (torch.randn(3000, 4, 16, generator=gen, device=device) for _ in range(2))
    ref, size = _exact(g, u, v)
    for got in (ops.gsddmm_u_dot_v(u, v, g),
                torch.ops.my_ops.gsddmm_u_dot_v(u, v, torch_boundary.script_graph(g))):
        assert bool(((got.double() - ref).abs() <= size * (16 * 2.0 ** -24)).all())


def test_first_call_inside_a_capture(device):
    """The destination column that the walk reads is not kept from a capture, where nothing
    has run yet: replays fill their own, eager calls build theirs."""
    rng = np.random.default_rng(4)
    n, e = 3000, 40_000
    g = prepare_graph(rng.integers(0, n, e), rng.integers(0, n, e), n, device=device)
    u, v = (torch.randn(n, 4, 16, device=device) for _ in range(2))
    assert not g.in_eid_is_identity and "in_rows" not in g._cache
    torch.cuda.synchronize()
    recorded = torch.cuda.CUDAGraph()
    with torch.cuda.graph(recorded):
        captured = ops.gsddmm_u_dot_v(u, v, g)
    assert "in_rows" not in g._cache
    eager = ops.gsddmm_u_dot_v(u, v, g)
    assert "in_rows" in g._cache
    ref = (u.double()[g.COO_src] * v.double()[g.COO_dst]).sum(2)
    assert float((eager.double() - ref).abs().max()) < 16 * 2.0 ** -23 * float(u.abs().max() * v.abs().max())
    for _ in range(3):
        captured.zero_()
        recorded.replay()
        torch.cuda.synchronize()
        assert torch.equal(captured, eager)
        assert torch.equal(ops.gsddmm_u_dot_v(u, v, g), eager)
