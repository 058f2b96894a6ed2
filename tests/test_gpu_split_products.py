"""fp32 products of the pair attention on the bf16 instruction (heads of 32 and 64 of 64
features): operands whose pieces do not cancel or lie far down in float's range, and the rows
of a tile that no pair owns."""
import numpy as np
import pytest
import torch

from graphiler_amd import capi, prepare_graph
from test_gpu_pair_attention import _by_pair

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


def _bits(word, *shape):
    return torch.full(shape, word, dtype=torch.int32).view(torch.float32)


@pytest.mark.parametrize("heads,d", [(1, 64), (2, 32)])
@pytest.mark.parametrize("values", ["cut", "near_one", "one_sign", "both_signs", "small", "tiny", "large"])
def test_products_against_float64(device, heads, d, values):
    """Pairs of one slot: the softmax weight is 1, the message is v @ M alone.  No sum is
    further from float64 than 2^-22 of the sum of its products' sizes: the products left out are
    below 2^-24 of theirs, the others are added in fp32 (the fp32 instruction's own 16 dependent
    sums are up to 6.2 x 2^-24 off on products of one sign).  Pieces that were cut off instead
    of rounded left out up to 7.8 x 2^-24, all of one sign, and third pieces out of bf16's range
    476 x 2^-24."""
    rng = np.random.default_rng(7)
    types, n = 3, 130
    dst = np.concatenate([np.arange(n), np.arange(64), np.arange(5)])
    et = np.repeat(np.arange(types), [n, 64, 5])
    g = prepare_graph(rng.integers(0, n, dst.size), dst, n, device=device, etype_of=et, num_etypes=types)
    normal = lambda *s: torch.from_numpy(rng.standard_normal(s, dtype=np.float32))
    v, msg = normal(n, heads * d), normal(types, heads, d, d)
    if values == "cut":                    # the most that cutting a significand in three loses
        v, msg = _bits(0x3f80ffff, n, heads * d), _bits(0x3f80ffff, types, heads, d, d)
    elif values == "near_one":             # significands around 1 + 2^-7
        v, msg = (1 + 2.0 ** -7 + 2.0 ** -8 * torch.sigmoid(x) for x in (v, msg))
    elif values == "one_sign":
        v, msg = v.abs(), msg.abs()
    elif values == "small":
        v = v * 2.0 ** -112
    elif values == "tiny":
        v, msg = v * 2.0 ** -118, msg * 2.0 ** 20
    elif values == "large":                # next to the largest float and what rounds past bf16's
        v, msg = _bits(0x7f7fffff, n, heads * d) * torch.sign(v), msg * 2.0 ** -20
    q, k = normal(n, heads * d) / d, normal(n, heads * d)
    att = normal(types, heads, d, d) / d ** 0.5
    m, _ = _tiles_pass(g, *(x.to(device) for x in (k, q, v, att, msg)))
    ref, _ = _by_pair(g, *(x.to(device) for x in (k, q, v, att, msg)))
    size, _ = _by_pair(g, *(x.to(device) for x in (k, q, v.abs(), att, msg.abs())))
    at = g.relation_pairs().by_type.cpu()
    err = (m.cpu().double() - ref[at]).abs() / size[at]
    assert float(err.max()) < 2.0 ** -22, f"{values}: {float(err.max()) * 2 ** 24:.2f} x 2^-24"


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
