"""fp32 products of the pair attention on the bf16 instruction (heads of 32 and 64 of 64
features): the rows of a tile that no pair owns."""
import numpy as np
import pytest
import torch

from graphiler_amd import capi, prepare_graph

pytestmark = pytest.mark.gpu


def _tiles_pass(g, k, q, v, att, msg):
    """(m, lse) in by_type order of the pass over prepared tiles; att as `_one_pass` takes it."""
    pairs, lib = g.relation_pairs(), capi.load()
    types, heads, d = att.shape[:3]
    stream = torch.cuda.current_stream().cuda_stream
    nbytes = lib.ga_pair_weights_bytes(types, heads, d, capi.GA_F32)
    assert nbytes > 0
    a, b = (torch.empty(nbytes, dtype=torch.uint8, device=k.device) for _ in range(2))
    capi.check(lib.ga_pair_weights(att.transpose(2, 3).contiguous().data_ptr(), None, capi.GA_F32, 1.0,
                                   msg.data_ptr(), a.data_ptr(), b.data_ptr(), types, heads, d, stream),
               "weights")
    m = torch.empty(pairs.num_pairs, heads * d, device=k.device)
    lse = torch.empty(pairs.num_pairs, heads, device=k.device)
    capi.check(lib.ga_pair_attention_tiles(
        pairs.rows.data_ptr(), pairs.tiles.data_ptr(), types, g.in_node_indices.data_ptr(),
        q.data_ptr(), k.data_ptr(), v.data_ptr(), a.data_ptr(), b.data_ptr(), m.data_ptr(),
        lse.data_ptr(), pairs.num_pairs, g.num_nodes, pairs.max_slots, heads, d, capi.GA_F32, stream),
        "tiles")
    return m, lse


@pytest.mark.parametrize("heads,d", [(1, 64), (2, 32)])
def test_rows_that_no_pair_owns(device, heads, d):
    """A tile with fewer than 64 pairs gives every pair the same bits as a full one: its other
    rows hold values that do not send the product to the fp32 instruction."""
    rng = np.random.default_rng(5)
    n, counts = 64, list(range(1, 64))
    src = rng.integers(0, n, (n, 3))
    dst = np.repeat(np.arange(n), 3)
    g = prepare_graph(np.concatenate([src.ravel()] + [src[:c].ravel() for c in counts]),
                      np.concatenate([dst] + [dst[:3 * c] for c in counts]), n, device=device,
                      etype_of=np.repeat(np.arange(64), [3 * c for c in [n] + counts]), num_etypes=64)
    rand = lambda *s: torch.from_numpy(rng.standard_normal(s, dtype=np.float32)).to(device)
    k, q, v = (rand(n, heads * d) for _ in range(3))
    att, msg = (rand(1, heads, d, d).expand(64, -1, -1, -1).contiguous() / d ** 0.5 for _ in range(2))
    m, lse = _tiles_pass(g, k, q, v, att, msg)
    at = n
    for c in counts:
        assert torch.equal(lse[:c], lse[at:at + c]), f"{c} pairs"
        assert torch.equal(m[:c], m[at:at + c]), f"{c} pairs"
        at += c
    assert at == m.shape[0]
