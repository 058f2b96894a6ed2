"""Graph preparation: uploads in page-locked pieces and pointers of sorted type columns,
against numpy."""
import numpy as np
import pytest
import torch

from graphiler_amd import prepare_graph
from graphiler_amd import graph as G

pytestmark = pytest.mark.gpu


# a piece holds 524,288 ids; arrays below 131,072 ids go over directly; the ring has three
@pytest.mark.parametrize("sizes", [(0,), (1, 131_071, 131_072), (524_288, 524_289),
                                   (2_000_003, 5, 1_700_000)])
def test_upload(device, sizes):
    rng = np.random.default_rng(sum(sizes))
    arrays = [rng.integers(-2 ** 62, 2 ** 62, n) for n in sizes]
    for got, want in zip(G._upload(arrays, device), arrays):
        assert got.dtype == torch.int64 and np.array_equal(got.cpu().numpy(), want)


@pytest.mark.parametrize("n,keys", [(0, 5), (1, 1), (255, 3), (257, 1000), (100_000, 7), (70_000, 70_001)])
def test_sorted_pointer(device, n, keys):
    rng = np.random.default_rng(n + keys)
    key = np.sort(rng.integers(0, keys, n)).astype(np.int64)
    pointer, status = G._sorted_pointer(torch.from_numpy(key).to(device), keys)
    assert status.tolist() == [0, 0]
    assert np.array_equal(pointer.cpu().numpy(), np.searchsorted(key, np.arange(keys + 1)))
    if n > 2:
        for at, value, want in ((n - 1, keys, [1, 0]), (0, -1, [1, 0]), (n // 2, -5, [1, 1])):
            bad = key.copy()
            bad[at] = value
            assert G._sorted_pointer(torch.from_numpy(bad).to(device), keys)[1].tolist() == want


@pytest.mark.parametrize("n,e", [(7, 20), (3000, 140_000), (9000, 600_000)])
def test_typed_graph(device, n, e):
    rng = np.random.default_rng(e)
    src, dst = rng.integers(0, n, e), rng.integers(0, n, e)
    nt, et = np.sort(rng.integers(0, 4, n)), np.sort(rng.integers(1, 30, e))
    g = prepare_graph(src, dst, n, device=device, ntype_of=nt, num_ntypes=5, etype_of=et, num_etypes=31)
    want = G.build_graph_arrays(src, dst, n)
    for name in ("in_pointer", "in_node_indices", "in_edge_indices", "out_pointer",
                 "out_node_indices", "out_edge_indices", "COO_src", "COO_dst"):
        assert np.array_equal(getattr(g, name).cpu().numpy(), getattr(want, name)), name
    assert np.array_equal(g.ntype_pointer.cpu().numpy(), G.type_pointer(nt, 5))
    assert np.array_equal(g.etype_pointer.cpu().numpy(), G.type_pointer(et, 31))
    assert np.array_equal(g.ntype_COO.cpu().numpy(), nt) and np.array_equal(g.etype_COO.cpu().numpy(), et)
    typed = dict(ntype_of=nt, num_ntypes=5, etype_of=et, num_etypes=31)
    with pytest.raises(ValueError, match="endpoint"):       # reported before a bad type
        prepare_graph(np.where(np.arange(e) == 3, n, src), dst, n, device=device, **{**typed, "etype_of": et[::-1]})
    with pytest.raises(ValueError, match="sorted by type"):
        prepare_graph(src, dst, n, device=device, **{**typed, "etype_of": et[::-1]})
    with pytest.raises(ValueError, match="type outside"):
        prepare_graph(src, dst, n, device=device, **{**typed, "num_ntypes": int(nt.max())})
    with pytest.raises(RuntimeError, match="one entry per node"):
        prepare_graph(src, dst, n, device=device, **{**typed, "ntype_of": nt[1:]})


@pytest.mark.parametrize("key,keys", [([], 4096), ([], 5000), ([0], 4096), ([4095], 4097), ([3, 3, 4096], 4097),
                                      ([7, 19_000_000], 20_000_000)])
def test_sorted_pointer_of_few_items(device, key, keys):
    """Far more keys than items: no lane walks a long gap by itself (20 M entries written one
    by one take tens of milliseconds, searched they are a launch)."""
    want = np.searchsorted(key, np.arange(keys + 1))
    column = torch.tensor(key, dtype=torch.int64, device=device)
    G._sorted_pointer(column, keys)
    start, end = (torch.cuda.Event(enable_timing=True) for _ in range(2))
    start.record()
    pointer, status = G._sorted_pointer(column, keys)
    end.record()
    assert status.tolist() == [0, 0] and np.array_equal(pointer.cpu().numpy(), want)
    assert start.elapsed_time(end) < 5.0


# tiles of 2,048 (up to 700,000 items) and 4,096 items, digits of up to ten bits: one, two and
# three passes; the library's sort above 16,777,216 items is what the large graphs' tests run
@pytest.mark.parametrize("keys,n", [(1, 1), (2, 2048), (5, 2049), (1024, 4097), (1025, 70_000),
                                    (1 << 20, 33_000), ((1 << 20) + 1, 33_001), ((1 << 30) + 7, 2047),
                                    (94_806, 700_000), (94_806, 700_001), (3000, 1_000_003)])
@pytest.mark.parametrize("kind", ["uniform", "hub", "ends"])
def test_grouping_is_a_stable_sort(device, keys, n, kind):
    rng = np.random.default_rng(n)
    src, dst = rng.integers(0, keys, n), rng.integers(0, keys, n)
    if kind == "hub":
        dst[rng.random(n) < 0.9] = keys // 2
    elif kind == "ends":
        src, dst = (keys - 1) * rng.integers(0, 2, n), np.full(n, keys - 1)
    dev = [torch.from_numpy(a).to(device) for a in (src, dst)]
    status = torch.empty(2, dtype=torch.int32, device=device)
    sides = G._group_both(*dev, keys, status) if keys <= 1 << 21 else \
        [G.group_on_device(dev[1], dev[0], keys)[:3], G.group_on_device(dev[0], dev[1], keys)[:3]]
    for (pointer, nbr, eid), key, other in zip(sides, (dst, src), (src, dst)):
        order = np.argsort(key, kind="stable")
        assert np.array_equal(eid.cpu().numpy(), order)
        assert np.array_equal(nbr.cpu().numpy(), other[order])
        at = np.unique(rng.integers(0, keys + 1, 1000))
        want = np.searchsorted(key[order], at)
        assert np.array_equal(pointer[torch.from_numpy(at).to(device)].cpu().numpy(), want)
    if keys <= 1 << 21:
        assert status.tolist() == [0, 0]
        for bad, want in ((0, [0, 1]), (1, [1, 0])):
            dev[bad][n // 2] = keys if bad else -1
            G._group_both(*dev, keys, status)
            assert status.tolist() == want
            dev[bad][n // 2] = 0


# a piece holds 1,048,576 ids, columns below 65,536 go over directly, and a column with a value
# that 32 bits do not hold goes over whole
@pytest.mark.parametrize("sizes", [(65_535, 65_536), (1_048_576, 1_048_577, 70_000, 3_300_000)])
@pytest.mark.parametrize("odd", [None, 2 ** 31, -2 ** 31 - 1, 2 ** 40 + 5])
def test_upload_of_ids(device, sizes, odd):
    rng = np.random.default_rng(sum(sizes))
    arrays = [rng.integers(-2 ** 31, 2 ** 31, n) for n in sizes]
    if odd is not None:
        for a in arrays:
            a[-1] = odd
    for got, want in zip(G._upload(arrays, device), arrays):
        assert got.dtype == torch.int64 and np.array_equal(got.cpu().numpy(), want)


def test_ids_beyond_32_bits_are_reported(device):
    n = 100_000
    src = np.arange(n) % 50
    bad = src.copy()
    bad[7] += 2 ** 32            # a valid id in its lower half
    for s, d in ((bad, src), (src, bad)):
        with pytest.raises(ValueError, match="endpoint"):
            prepare_graph(s, d, 50, device=device)
    types = np.sort(src) * 0
    types[-1] = 2 ** 32
    with pytest.raises(ValueError, match="type outside"):
        prepare_graph(src, src, 50, device=device, etype_of=types, num_etypes=3)


@pytest.mark.parametrize("n", [1, 255, 256, 257, 3000])
def test_in_degrees(device, n):
    from graphiler_amd import ops
    rng = np.random.default_rng(n)
    dst = rng.integers(0, n, 2 * n) // 2
    g = prepare_graph(rng.integers(0, n, 2 * n), dst, n, device=device)
    want = np.bincount(dst, minlength=n).astype(np.float32)[:, None]
    assert np.array_equal(ops.in_degrees(g).cpu().numpy(), want)
    assert np.array_equal(ops.in_degrees(g, at_least=1).cpu().numpy(), np.maximum(want, 1))
