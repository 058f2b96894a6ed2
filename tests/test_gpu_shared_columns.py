"""Row reductions whose lane groups read the slot-indexed columns for one another
(groups of 8 lanes and of 16 and more), dense graphs with tables of several times an L2,
and the short runs of small graphs: widths around the lane counts where the layouts change, against the oracle."""
import numpy as np
import pytest
import torch

import oracle
from graphiler_amd import ops, prepare_graph
from graphiler_amd.graph import build_graph_arrays
from helpers import TOL_BF16, TOL_F32, assert_close, skewed_graph, to_bf16_f32

pytestmark = pytest.mark.gpu


def _dev(a, device, bf16=False):
    t = torch.from_numpy(np.ascontiguousarray(a)).to(device)
    return t.to(torch.bfloat16) if bf16 else t


# edges: one slot, less than / exactly / just over a batch of eight, runs of 8, 16 and 32 slots
@pytest.mark.parametrize("edges", [1, 7, 8, 9, 1000, 9001, 40_003])
@pytest.mark.parametrize("feat", [17, 28, 32, 36, 48, 64, 65, 100, 132, 260])
@pytest.mark.parametrize("bf16", [False, True])
def test_widths_and_run_lengths(device, edges, feat, bf16):
    rng = np.random.default_rng(edges * 7 + feat)
    n = 300
    src, dst = skewed_graph(rng, n, edges - edges // 3, edges // 3)
    g = prepare_graph(src, dst, n, device=device)
    arr = build_graph_arrays(src, dst, n)
    adj = (arr.in_pointer, arr.in_node_indices, arr.in_edge_indices)
    tol = TOL_BF16 if bf16 else TOL_F32
    x = rng.standard_normal((n, feat), dtype=np.float32)
    xe = rng.standard_normal((edges, feat), dtype=np.float32)
    w = rng.standard_normal((edges, 1), dtype=np.float32)
    el, er = (rng.standard_normal((n, 1), dtype=np.float32) for _ in range(2))
    if bf16:
        x, xe = to_bf16_f32(x), to_bf16_f32(xe)
    dx, dxe, dw = _dev(x, device, bf16), _dev(xe, device, bf16), _dev(w, device)
    what = f"E={edges} F={feat} bf16={bf16}"
    host = lambda t: t.float().cpu().numpy()
    for reduce in ("sum", "max"):
        ref = oracle.spmm(*adj, x, op="copy_u", reduce=reduce)
        assert_close(host(ops.spmm(g, "copy_u", reduce, dx)), ref, tol, f"copy_u {reduce} {what}")
    ref = oracle.spmm(*adj, xe, op="copy_e")
    assert_close(host(ops.spmm(g, "copy_e", "sum", dxe)), ref, tol, f"copy_e {what}")
    ref = oracle.spmm(*adj, x, w, op="u_mul_e")
    assert_close(host(ops.spmm(g, "u_mul_e", "sum", dx, dw)), ref, tol, f"u_mul_e {what}")
    scale = rng.standard_normal(n).astype(np.float32)
    ref = np.maximum(oracle.spmm(*adj, x) * scale[:, None], 0)
    got = ops.spmm_scaled(dx, g, row_scale=_dev(scale, device), activation="relu")
    assert_close(host(got), ref, tol, f"scaled {what}")
    ref = oracle.gat_aggregate(arr.in_pointer, arr.in_node_indices, el, er, x, heads=1, slope=0.2)
    got = ops.gat_aggregate(_dev(el, device), _dev(er, device), dx, g, 0.2)
    assert_close(host(got), ref, tol, f"gat {what}")
    logit = rng.standard_normal((edges, 1), dtype=np.float32)
    logit[rng.random((edges, 1)) < 0.1] = -1e30       # masked edges weigh nothing
    a = oracle.segment_softmax(arr.in_pointer, arr.in_edge_indices, logit)
    ref = oracle.spmm(*adj, (xe * a).astype(np.float32), op="copy_e")
    got = ops.edge_softmax_sum(_dev(logit, device), dxe, g)
    assert_close(host(got), ref, tol, f"softmax sum {what}")


@pytest.mark.parametrize("heads,dim", [(2, 64), (2, 32), (4, 128), (2, 128), (8, 8), (3, 64)])
@pytest.mark.parametrize("bf16", [False, True])
def test_heads_with_and_without_a_shared_batch(device, heads, dim, bf16):
    rng = np.random.default_rng(heads * dim)
    n, edges = 400, 7000
    src, dst = skewed_graph(rng, n, 5000, 2000)
    g = prepare_graph(src, dst, n, device=device)
    arr = build_graph_arrays(src, dst, n)
    adj = (arr.in_pointer, arr.in_node_indices, arr.in_edge_indices)
    x = rng.standard_normal((n, heads * dim), dtype=np.float32)
    x = to_bf16_f32(x) if bf16 else x
    tol = TOL_BF16 if bf16 else TOL_F32
    w = rng.standard_normal((edges, heads), dtype=np.float32)
    el, er = (rng.standard_normal((n, heads), dtype=np.float32) for _ in range(2))
    dx = _dev(x, device, bf16)
    ref = oracle.spmm(*adj, x, w, op="u_mul_e", heads=heads)
    got = ops.spmm(g, "u_mul_e", "sum", dx.view(n, heads, dim), _dev(w, device).view(edges, heads, 1))
    assert_close(got.float().cpu().numpy().reshape(n, -1), ref.reshape(n, -1), tol, "u_mul_e")
    ref = oracle.gat_aggregate(arr.in_pointer, arr.in_node_indices, el, er, x, heads=heads, slope=0.2)
    got = ops.gat_aggregate(_dev(el, device), _dev(er, device), dx, g, 0.2)
    assert_close(got.float().cpu().numpy().reshape(n, -1), ref.reshape(n, -1), tol, "gat")


# rows over one run of eight slots, over as many runs as a word of flags has bits and one less
# and more, over all runs of a workgroup: the chain inside a workgroup from every lane-group width
@pytest.mark.parametrize("feat", [1, 3, 5, 8, 12, 20, 64, 100])
@pytest.mark.parametrize("bf16", [False, True])
def test_rows_over_many_runs(device, feat, bf16):
    rng = np.random.default_rng(feat)
    lengths = np.array([1, 7, 8, 9, 16, 17, 31, 33, 503, 511, 512, 513, 520, 1017, 1024, 1033,
                        1543, 2040, 2048, 2049, 5000, 0, 3, 64 * 8 + 4, 2, 127])
    lengths = np.concatenate([rng.permutation(lengths), rng.permutation(lengths)])
    n, edges = lengths.size, int(lengths.sum())
    dst = np.repeat(np.arange(n), lengths)
    src = rng.integers(0, n, edges)
    g = prepare_graph(src, dst, n, device=device)
    arr = build_graph_arrays(src, dst, n)
    adj = (arr.in_pointer, arr.in_node_indices, arr.in_edge_indices)
    x = rng.standard_normal((n, feat), dtype=np.float32)
    x = to_bf16_f32(x) if bf16 else x
    el, er = (rng.standard_normal((n, 1), dtype=np.float32) for _ in range(2))
    dx, tol = _dev(x, device, bf16), TOL_BF16 if bf16 else TOL_F32
    host = lambda t: t.float().cpu().numpy()
    for reduce in ("sum", "max"):
        ref = oracle.spmm(*adj, x, op="copy_u", reduce=reduce)
        assert_close(host(ops.spmm(g, "copy_u", reduce, dx)), ref, tol, f"{reduce} F={feat}")
    ref = oracle.gat_aggregate(arr.in_pointer, arr.in_node_indices, el, er, x, heads=1, slope=0.2)
    got = ops.gat_aggregate(_dev(el, device), _dev(er, device), dx, g, 0.2)
    assert_close(host(got), ref, tol, f"gat F={feat}")


# 32 edges per node and a table of 16 MB, several times an L2
@pytest.mark.parametrize("feat,bf16", [(64, False), (128, False), (192, True), (256, True)])
def test_dense_graph_with_a_large_table(device, feat, bf16):
    rng = np.random.default_rng(feat)
    n = (16 << 20) // (feat * (2 if bf16 else 4)) + 1
    edges = 32 * n
    src, dst = skewed_graph(rng, n, edges - 50_000, 50_000)
    g = prepare_graph(src, dst, n, device=device)
    arr = build_graph_arrays(src, dst, n)
    x = rng.standard_normal((n, feat), dtype=np.float32)
    x = to_bf16_f32(x) if bf16 else x
    adj = (arr.in_pointer, arr.in_node_indices, arr.in_edge_indices)
    ref = oracle.spmm(*adj, x)
    dx = _dev(x, device, bf16)
    got = ops.SpMMSrc(dx, [1], False, None, g).float().cpu().numpy()
    assert_close(got, ref, TOL_BF16 if bf16 else TOL_F32, f"large table F={feat}")
    scale = rng.standard_normal(n).astype(np.float32)
    got = ops.spmm_scaled(dx, g, row_scale=_dev(scale, device), activation="relu")
    assert_close(got.float().cpu().numpy(), np.maximum(ref * scale[:, None], 0),
                 TOL_BF16 if bf16 else TOL_F32, f"large table, scaled F={feat}")
