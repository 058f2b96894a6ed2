"""Sums over slots ordered by source classes against the plain sum and float64."""
import gc

import numpy as np
import pytest
import torch

from graphiler_amd import capi, ops, prepare_graph


def _degrees(deg):
    deg = np.asarray(deg, np.int64)
    deg = deg[deg > 0]
    b = np.floor(np.log2(deg)).astype(np.int64)
    return (np.bincount(b, minlength=capi.GA_DEGREE_BUCKETS).astype(np.int64),
            np.bincount(b, deg, minlength=capi.GA_DEGREE_BUCKETS).astype(np.int64))


def _classes(deg, n, e, feat, dt):
    nodes, edges = _degrees(deg)
    return capi.load().ga_spmm_source_classes(nodes.ctypes.data, edges.ctypes.data, n, e, feat, dt)


def test_rule_on_the_host():
    lib = capi.load()
    even = np.full(100_000, 200)
    assert _classes(even, 100_000, 20_000_000, 64, capi.GA_F32) == 8
    assert _classes(even, 100_000, 20_000_000, 64, capi.GA_BF16) == 4
    # nearly all gathers go to rows that an L2 holds anyway
    hubs = np.where(np.arange(100_000) < 2_000, 9_900, 2)
    assert _classes(hubs, 100_000, int(hubs.sum()), 64, capi.GA_F32) == 0
    # few edges per node; a table an L2 holds; rows that 16-byte accesses do not tile
    for n, e, feat in ((100_000, 1_500_000, 64), (10_000, 2_000_000, 64), (100_000, 20_000_000, 66),
                       (100_000, 20_000_000, 4), (0, 0, 64), (1 << 29, (1 << 31) - 1, 64)):
        assert lib.ga_spmm_source_classes(None, None, n, e, feat, capi.GA_F32) == 0


def _graph(n, e, seed, hub=False):
    rng = np.random.default_rng(seed)
    src, dst = rng.integers(0, n, e), rng.integers(0, n, e)
    if hub:
        dst[: e // 2] = n // 2
    return prepare_graph(src, dst, n, device="cuda:0")


def _sum64(g, x):
    out = torch.zeros(g.num_nodes, x.shape[1], dtype=torch.float64, device="cuda")
    return out.index_add_(0, g.COO_dst, x.double()[g.COO_src])


def _run(g, x, classes, scale=None, act=0):
    lib = capi.load()
    from graphiler_amd.graph import _build_source_classes
    c = _build_source_classes(g, classes)
    out = torch.full_like(x, float("nan"))
    dt = capi.GA_F32 if x.dtype == torch.float32 else capi.GA_BF16
    n = lib.ga_spmm_classes_workspace_bytes(g.num_nodes, g.num_edges, x.shape[1], classes)
    ws = torch.full((n // 4,), float("nan"), device="cuda")
    args = [c.pointer.data_ptr(), c.rows.data_ptr(), c.nbr.data_ptr(), x.data_ptr(), out.data_ptr(),
            None if scale is None else scale.data_ptr(), act, g.num_nodes, g.num_edges, x.shape[1],
            classes, dt, ws.data_ptr(), n, torch.cuda.current_stream().cuda_stream]
    assert lib.ga_spmm_classes(*args[:-2], n - 4, args[-1]) == capi.GA_EWORKSPACE
    capi.check(lib.ga_spmm_classes(*args), "ga_spmm_classes")
    return c, out


# one unit of the partition holds 4096 slots, a block of source ids 64; the widths are the
# lane groups of the three builds and a second feature tile
@pytest.mark.gpu
@pytest.mark.parametrize("n,e,hub", [(1, 1, False), (70, 4095, False), (500, 4097, True),
                                     (3000, 40_000, True), (20_011, 200_003, False)])
@pytest.mark.parametrize("classes", [2, 4, 8])
@pytest.mark.parametrize("dtype,feat", [(torch.float32, 8), (torch.float32, 20), (torch.float32, 64),
                                        (torch.float32, 260), (torch.bfloat16, 16),
                                        (torch.bfloat16, 136)])
def test_sums_and_layout(n, e, hub, classes, dtype, feat):
    g = _graph(n, e, 11 * n + classes, hub)
    gen = torch.Generator(device="cuda").manual_seed(feat)
    x = torch.randn(n, feat, generator=gen, device="cuda").to(dtype)
    scale = torch.rand(n, generator=gen, device="cuda") + 0.5
    c, out = _run(g, x, classes)
    # the layout: a stable partition by the class that every slot's key names
    src, rows = c.nbr.long(), c.rows.long()
    cls = torch.div(rows, n, rounding_mode="floor")
    want = ((((g.in_node_indices.long() >> 6) * 0x9E3779B1) & 0xFFFFFFFF) * classes) >> 32
    order = torch.argsort(want, stable=True)
    assert torch.equal(cls, want[order]) and torch.equal(src, g.in_node_indices.long()[order])
    assert torch.equal(rows - cls * n, g.in_row_of_slot.long()[order])
    assert torch.equal(c.pointer.long(),
                       torch.searchsorted(rows, torch.arange(classes * n + 1, device="cuda")))
    # fp32 sums of at most e terms: every addition rounds to 2^-24 of the running sum, bf16
    # results once more to 2^-8
    ref = _sum64(g, x)
    bound = _sum64(g, x.abs()) * (64 * 2.0 ** -24) + 1e-30
    if dtype == torch.bfloat16:
        bound += ref.abs() * 2.0 ** -8
    assert bool(((out.double() - ref).abs() <= bound).all())
    # the tail: what the separate operators give, bit for bit in fp32
    _, tail = _run(g, x, classes, scale, capi.GA_ACT_RELU)
    if dtype == torch.float32:
        assert torch.equal(tail, torch.relu(out * scale.unsqueeze(1)))
    else:
        err = (tail.double() - torch.relu(ref * scale.double().unsqueeze(1))).abs()
        assert bool((err <= 1.5 * bound + 2.0 ** -7 * ref.abs()).all())


@pytest.mark.gpu
def test_operators_take_the_order_where_it_is_faster():
    n, e = 40_000, 6_000_000
    g = _graph(n, e, 5)
    x = torch.randn(n, 64, device="cuda")
    scale = torch.rand(n, 1, device="cuda")
    # captured before any eager call: the plain sum, no layout is built inside the capture
    g.in_row_of_slot, g.in_eid_is_identity
    g.workspace(capi.load().ga_spmm_workspace_bytes(e, 64))
    torch.cuda.synchronize()
    hipgraph = torch.cuda.CUDAGraph()
    with torch.cuda.graph(hipgraph):
        captured = ops.SpMMSrc(x, [1], False, None, g)
    assert not any(isinstance(k, tuple) for k in g._cache)
    out = ops.SpMMSrc(x, [1], False, None, g)
    assert g.source_classes(64, capi.GA_F32).num_classes > 0
    ref = _sum64(g, x)
    bound = _sum64(g, x.abs()) * (64 * 2.0 ** -24)
    for _ in range(3):
        hipgraph.replay()
        torch.cuda.synchronize()
        assert bool(((captured.double() - ref).abs() <= bound).all())
        assert bool(((out.double() - ref).abs() <= bound).all())
        assert torch.equal(ops.spmm_scaled(x, g, scale, "relu"), torch.relu(out * scale))
    # captured with the layout in place
    again = torch.cuda.CUDAGraph()
    with torch.cuda.graph(again):
        captured = ops.SpMMSrc(x, [1], False, None, g)
    for _ in range(3):
        captured.zero_()
        again.replay()
        torch.cuda.synchronize()
        assert torch.equal(captured, out)
    # rows off a 16-byte boundary, the transposed sum and other reducers keep their routes
    shifted = torch.randn(n * 64 + 1, device="cuda")[1:].view(n, 64)
    err = (ops.SpMMSrc(shifted, [1], False, None, g).double() - _sum64(g, shifted)).abs()
    assert bool((err <= _sum64(g, shifted.abs()) * (64 * 2.0 ** -24)).all())


@pytest.mark.gpu
def test_boundary_operators_take_the_order_where_it_is_faster():
    from graphiler_amd import torch_boundary
    torch_boundary.load()
    n, e = 40_000, 6_000_000
    g = _graph(n, e, 6)
    t = torch.classes.my_classes.DGLGraph(
        g.in_pointer, g.in_node_indices, g.in_edge_indices, g.out_pointer, g.out_node_indices,
        g.out_edge_indices, g.COO_src, g.COO_dst, None, None)
    x = torch.randn(n, 64, device="cuda")
    scale = torch.rand(n, 1, device="cuda")
    assert torch.equal(torch.ops.my_ops.SpMMSrc(x, [1], False, None, t),
                       ops.SpMMSrc(x, [1], False, None, g))
    assert torch.equal(torch.ops.my_ops.SpMMScaled(x, scale, capi.GA_ACT_RELU, False, t),
                       ops.spmm_scaled(x, g, scale, "relu"))
    assert g.source_classes(64, capi.GA_F32).num_classes > 0


@pytest.mark.gpu
@pytest.mark.parametrize("lengths", [[1], [0, 0, 0], [1, 2, 3, 4, 7, 8, 0, 255, 256, 2 ** 20 + 1],
                                     list(range(257)), [2 ** 31 - 1], [3] * 300_001])
def test_degrees_counted_on_the_device(lengths):
    deg = np.asarray(lengths, np.int64)
    pointer = torch.from_numpy(np.concatenate([[0], np.cumsum(deg)]).astype(np.int32)).cuda()
    out = torch.full((2, capi.GA_DEGREE_BUCKETS), -1, dtype=torch.int64, device="cuda")
    capi.check(capi.load().ga_degree_buckets(pointer.data_ptr(), deg.size, out.data_ptr(),
                                             torch.cuda.current_stream().cuda_stream), "buckets")
    nodes, edges = _degrees(deg)
    assert (out.cpu().numpy() == np.stack([nodes, edges])).all()


@pytest.mark.gpu
def test_sums_of_dense_graphs_under_deterministic_algorithms():
    """Counting the degrees asks torch for nothing it refuses there."""
    from graphiler_amd import torch_boundary
    torch_boundary.load()
    g = _graph(40_000, 6_000_000, 7)
    t = torch_boundary.script_graph(g)
    x = torch.randn(40_000, 64, device="cuda")
    torch.use_deterministic_algorithms(True)
    try:
        out = ops.SpMMSrc(x, [1], False, None, g)
        same = torch.ops.my_ops.SpMMSrc(x, [1], False, None, t)
    finally:
        torch.use_deterministic_algorithms(False)
    assert g.source_classes(64, capi.GA_F32).num_classes > 0
    assert torch.equal(out, same)
    assert bool(((out.double() - _sum64(g, x)).abs() <= _sum64(g, x.abs()) * (64 * 2.0 ** -24)).all())


def _fill_free_blocks():
    """Tensors in every free block of more than a megabyte that torch holds: what is asked for from
    here on needs memory of the device, whatever earlier tests left between their allocations."""
    held = []
    for segment in torch.cuda.memory_snapshot():
        if segment["stream"] == 0 and tuple(segment["segment_pool_id"]) == (0, 0) and segment["segment_type"] == "large":
            held += [torch.empty(b["size"], dtype=torch.uint8, device="cuda") for b in segment["blocks"]
                     if b["state"] == "inactive" and b["size"] > 1 << 20]
    return held


@pytest.mark.gpu
@pytest.mark.parametrize("boundary", [False, True])
@pytest.mark.parametrize("used", [False, True])
def test_scratch_that_does_not_fit_is_asked_for_once(boundary, used):
    from graphiler_amd import torch_boundary
    torch_boundary.load()
    lib, n, e, feat = capi.load(), 40_000, 6_000_000, 512
    gc.collect()            # no large segment of earlier tests to take blocks from
    torch.cuda.empty_cache()
    g = _graph(n, e, 8)
    t = torch_boundary.script_graph(g)
    x = torch.randn(n, feat, device="cuda")
    call = (lambda y: torch.ops.my_ops.SpMMSrc(y, [1], False, None, t)) if boundary else \
        (lambda y: ops.SpMMSrc(y, [1], False, None, g))
    probe = _graph(n, e, 8)
    k = probe.source_classes(feat, capi.GA_F32).num_classes
    narrow = next(f for f in (256, 128, 64) if probe.source_classes(f, capi.GA_F32).num_classes == k)
    plain = lib.ga_spmm_workspace_bytes(e, feat)
    classes = lib.ga_spmm_classes_workspace_bytes(n, e, feat, k)
    del probe
    call(x.to(torch.float64).max(1).values.float().view(n, 1))      # row ids; no classes here
    if used:                # the layout serves another width and stays
        few = x[:, :narrow].contiguous()
        before = call(few)
    torch.cuda.synchronize()
    torch.cuda.empty_cache()
    reserved = torch.cuda.memory_reserved()
    held = _fill_free_blocks()
    assert torch.cuda.memory_reserved() == reserved
    total = torch.cuda.get_device_properties(0).total_memory
    room = 4 * n * feat * 2 + 10 * e + plain + (64 << 20)
    assert classes > room
    ooms = lambda: torch.cuda.memory_stats()["num_ooms"]
    try:
        torch.cuda.set_per_process_memory_fraction((torch.cuda.memory_reserved() + room) / total)
        at = ooms()
        first = call(x)
        assert ooms() == at + 1
        second = call(x)
        assert ooms() == at + 1
    finally:
        torch.cuda.set_per_process_memory_fraction(1.0)
    del held
    assert torch.equal(first, second)
    part = x[:, :16].contiguous()
    err = (first[:, :16].double() - _sum64(g, part)).abs()
    assert bool((err <= _sum64(g, part.abs()) * (64 * 2.0 ** -24)).all())
    if not boundary:
        assert (("classes", k) in g._cache) == used
    if used:
        assert torch.equal(call(few), before)
