"""The one-pass (destination, relation) pair attention of an HGT layer against float64:
tile edges (pairs per relation around 64), slots per pair around the batch of four, every
head layout it takes, and the pair size from which the separate passes run."""
import numpy as np
import pytest
import torch

from graphiler_amd import ops, prepare_graph, torch_boundary
from helpers import TOL_BF16, TOL_F32, assert_close

pytestmark = pytest.mark.gpu


def _typed_graph(rng, pairs_per_type, largest, device):
    """Relation t has pairs_per_type[t] destinations with 1 .. 9 edges, one has `largest`."""
    n = max(pairs_per_type) + 20
    src, dst, et = [], [], []
    for t, p in enumerate(pairs_per_type):
        who = rng.permutation(n)[:p]
        cnt = rng.integers(1, 10, p)
        cnt[:3] = [4, 5, 8][:min(3, p)]
        if t == 1 and p:
            cnt[-1] = largest
        dst.append(np.repeat(who, cnt))
        et.append(np.full(cnt.sum(), t))
    dst, et = np.concatenate(dst), np.concatenate(et)
    src = rng.integers(0, n, dst.size)
    g = prepare_graph(src, dst, n, device=device, etype_of=et, num_etypes=len(pairs_per_type))
    return g, src, dst, et, n


@pytest.mark.parametrize("heads,d", [(1, 64), (2, 32), (4, 16), (8, 8), (2, 64), (4, 32), (8, 16), (16, 8)])
@pytest.mark.parametrize("bf16", [False, True])
@pytest.mark.parametrize("largest", [9, 256, 257])
def test_against_float64(device, heads, d, bf16, largest):
    rng = np.random.default_rng(heads * d + largest)
    per = [64, 65, 1, 0, 63, 300, 129]
    g, src, dst, et, n = _typed_graph(rng, per, largest, device)
    assert g.relation_pairs().max_slots == largest and g.relation_pairs().num_pairs == sum(per)
    dt = torch.bfloat16 if bf16 else torch.float32
    rand = lambda *s: torch.from_numpy(rng.standard_normal(s, dtype=np.float32)).to(dt)
    k, q, v = (rand(n, heads * d) for _ in range(3))
    att, msg = (rand(len(per), heads, d, d) / d ** 0.5 for _ in range(2))
    k[::7] *= 6                       # scores spread over tens: the running maximum moves
    factor = 1.0 / d ** 0.5
    got = ops.relation_pair_attention(*(x.to(device) for x in (k, q, v, att, msg)), None, g,
                                      factor=factor)
    w = lambda x, rows: torch.einsum("ehk,ehkm->ehm", x.double().view(n, heads, d)[rows], _pick)
    s, t, r = (torch.from_numpy(np.asarray(a)) for a in (src, et, dst))
    _pick = att.double()[t]
    score = (w(k, s) * q.double().view(n, heads, d)[r]).sum(2) * factor
    _pick = msg.double()[t]
    msgs = w(v, s)
    top = torch.full((n, heads), -np.inf, dtype=torch.float64).index_reduce_(0, r, score, "amax")
    p = torch.exp(score - top[r])
    den = torch.zeros(n, heads, dtype=torch.float64).index_add_(0, r, p)
    ref = torch.zeros(n, heads, d, dtype=torch.float64).index_add_(0, r, (p / den[r]).unsqueeze(2) * msgs)
    # scores of tens in bf16 queries move by a rounding (2^-9 of tens), which the weights show
    tol = 2 * TOL_BF16 if bf16 else 2 * TOL_F32
    assert_close(got.float().cpu().numpy(), ref.reshape(n, -1).numpy(), tol, f"{heads}x{d} bf16={bf16}")
    torch_boundary.load()
    same = torch.ops.my_ops.relation_pair_attention(
        *(x.to(device) for x in (k, q, v, att, msg)), None, 1.0 / factor, torch_boundary.script_graph(g))
    if g.num_edges >= 2 * sum(per):
        assert torch.equal(got, same)
