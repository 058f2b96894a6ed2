"""Operators that gather rows by node id refuse tensors with fewer rows than the graph has nodes."""
import numpy as np
import pytest
import torch

from graphiler_amd import layers, ops, prepare_graph

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("short", [0, 1, 2])
def test_a_row_for_every_node(device, short):
    n, rng = 40, np.random.default_rng(2)
    g = prepare_graph(rng.integers(0, n, 200), rng.integers(0, n, 200), n, device=device)
    rows = lambda i: n - 1 if i == short else n
    el, er, z = (torch.randn(rows(i), w, device=device) for i, w in enumerate((4, 4, 64)))
    with pytest.raises(RuntimeError, match="one row per node"):
        ops.gat_aggregate(el, er, z, g)
    if short > 0:
        with pytest.raises(RuntimeError, match="one row per node"):
            ops.gat_aggregate_from_z(torch.randn(4, 16, device=device), er, z, g)
    if short < 2:
        with pytest.raises(RuntimeError, match="one row per node"):
            ops.gsddmm_u_add_v_mul_alpha(el, er, 1, g)
        with pytest.raises(RuntimeError, match="one row per node"):
            ops.gsddmm_u_dot_v(el, er, g)


def test_a_layer_refuses_fewer_rows(device):
    n, rng = 40, np.random.default_rng(3)
    g = prepare_graph(rng.integers(0, n, 200), rng.integers(0, n, 200), n, device=device)
    x, w, a = (torch.randn(*s, device=device) for s in ((n - 1, 20), (20, 64), (2, 4, 16)))
    with pytest.raises(RuntimeError, match="one row per node"):
        layers.gat_layer(g, x, w, a, 4)
    with pytest.raises(RuntimeError, match="one row per node"):
        layers.gat_layer(g, x, w, a, 4, fused=False)
