"""The one-pass (destination, relation) pair attention of an HGT layer against float64:
tile edges (pairs per relation around 64), slots per pair around the batch of four, every
head layout it takes, the largest pair it takes, and lists of more than a million pairs.
The layer's operator takes the pass or three launches by a rule; the pass is also called
by itself, so that it is the pass that is checked."""
import numpy as np
import pytest
import torch

from graphiler_amd import capi, ops, prepare_graph, torch_boundary
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


def _one_pass(g, k, q, v, att, msg, max_slots=None):
    """(return code, m, lse) of ga_pair_attention: pairs in slot order, `att` as the query
    side needs it (transposed)."""
    pairs, heads, d = g.relation_pairs(), att.shape[1], att.shape[2]
    m = torch.empty(pairs.num_pairs, heads * d, dtype=k.dtype, device=k.device)
    lse = torch.empty(pairs.num_pairs, heads, device=k.device)
    rc = capi.load().ga_pair_attention(
        pairs.type_pointer.data_ptr(), g.num_etypes, pairs.by_type.data_ptr(),
        pairs.dst_by_type.data_ptr(), pairs.pair_pointer.data_ptr(), g.in_node_indices.data_ptr(),
        q.data_ptr(), k.data_ptr(), v.data_ptr(), att.data_ptr(), msg.data_ptr(), m.data_ptr(),
        lse.data_ptr(), pairs.num_pairs, pairs.max_slots if max_slots is None else max_slots, heads,
        d, capi.GA_F32 if k.dtype == torch.float32 else capi.GA_BF16,
        torch.cuda.current_stream().cuda_stream)
    return rc, m, lse


def _by_pair(g, k, q, v, att, msg):
    """The same in float64 on the CPU."""
    pairs, heads, d = g.relation_pairs(), att.shape[1], att.shape[2]
    host = lambda t: t.cpu().double() if t.is_floating_point() else t.cpu().long()
    k, q, v, att, msg = (host(t) for t in (k, q, v, att, msg))
    P, src, pair = pairs.num_pairs, host(g.in_node_indices), host(pairs.pair_of_slot)
    kind = torch.empty(P, dtype=torch.int64)
    kind[host(pairs.by_type)] = torch.repeat_interleave(
        torch.arange(g.num_etypes), torch.diff(host(pairs.type_pointer)))
    rows = lambda x, at: x.view(-1, heads, d)[at]
    qp = torch.einsum("phk,phkm->phm", rows(q, host(pairs.pair_dst)), att[kind])
    score = (rows(k, src) * qp[pair]).sum(2)
    top = torch.full((P, heads), -np.inf, dtype=torch.float64).index_reduce_(0, pair, score, "amax")
    p = torch.exp(score - top[pair])
    den = torch.zeros(P, heads, dtype=torch.float64).index_add_(0, pair, p)
    vp = torch.zeros(P, heads, d, dtype=torch.float64).index_add_(
        0, pair, (p / den[pair]).unsqueeze(2) * rows(v, src))
    return torch.einsum("phk,phkm->phm", vp, msg[kind]).reshape(P, -1), top + torch.log(den)


@pytest.mark.parametrize("heads,d", [(1, 64), (2, 32), (4, 16), (8, 8), (2, 64), (4, 32), (8, 16), (16, 8)])
@pytest.mark.parametrize("bf16", [False, True])
def test_the_pass_by_itself(device, heads, d, bf16):
    rng = np.random.default_rng(heads * d + bf16)
    per = [64, 65, 1, 0, 63, 300, 129]
    g, *_, n = _typed_graph(rng, per, 256, device)
    dt = torch.bfloat16 if bf16 else torch.float32
    rand = lambda *s: torch.from_numpy(rng.standard_normal(s, dtype=np.float32)).to(device).to(dt)
    k, q, v = (rand(n, heads * d) for _ in range(3))
    att, msg = (rand(len(per), heads, d, d) / d ** 0.5 for _ in range(2))
    k[::7] *= 4
    rc, m, lse = _one_pass(g, k, q / d ** 0.5, v, att, msg)
    assert rc == capi.GA_OK
    assert _one_pass(g, k, q, v, att, msg, max_slots=257)[0] == capi.GA_EUNSUPPORTED
    ref_m, ref_lse = _by_pair(g, k, q / d ** 0.5, v, att, msg)
    # a score is a sum of d products of a bf16-rounded query (2^-9 of it): tens of them move
    # the weights by what the operator's test allows
    tol = 2 * TOL_BF16 if bf16 else 2 * TOL_F32
    assert_close(m.float().cpu().numpy(), ref_m.numpy(), tol, f"m {heads}x{d} bf16={bf16}")
    assert_close(lse.cpu().numpy(), ref_lse.numpy(), tol, f"lse {heads}x{d} bf16={bf16}")


@pytest.mark.parametrize("heads,d,bf16", [(1, 64, False), (8, 16, True), (2, 64, False)])
def test_scores_that_are_not_finite(device, heads, d, bf16):
    """The pass and the three launches agree where scores are +inf, -inf or NaN."""
    rng = np.random.default_rng(3)
    g, *_, n = _typed_graph(rng, [64, 65, 1, 0, 63, 300, 129], 40, device)
    dt = torch.bfloat16 if bf16 else torch.float32
    rand = lambda *s: torch.from_numpy(rng.standard_normal(s, dtype=np.float32)).to(device).to(dt)
    k, q, v = (rand(n, heads * d) for _ in range(3))
    att, msg = (rand(7, heads, d, d) / d ** 0.5 for _ in range(2))
    k[5, :] = float("nan")
    k[11, 0], k[17, 0] = float("inf"), -float("inf")
    rc, m, lse = _one_pass(g, k, q, v, att, msg)
    assert rc == capi.GA_OK
    pairs, lib, stream = g.relation_pairs(), capi.load(), torch.cuda.current_stream().cuda_stream
    P, E, code = pairs.num_pairs, g.num_edges, capi.GA_BF16 if bf16 else capi.GA_F32

    def typed_rows(x, index, w):
        y = torch.empty(P, heads * d, dtype=dt, device=device)
        capi.check(lib.ga_segment_mm_gather(
            pairs.type_pointer.data_ptr(), g.num_etypes, x.data_ptr(), index.data_ptr(), w.data_ptr(),
            y.data_ptr(), None, None, None, None, None, P, heads, d, d, code, stream), "rows")
        return y

    ws = g.workspace(max(lib.ga_gat_workspace_bytes(i, heads * d, heads) for i in (E, P)))
    q_pair, v_pair = typed_rows(q, pairs.dst_by_type, att), torch.empty_like(m)
    lse3 = torch.empty_like(lse)
    capi.check(lib.ga_dot_attention_sum(
        pairs.pair_pointer.data_ptr(), pairs.pair_of_slot.data_ptr(), g.in_node_indices.data_ptr(),
        pairs.rank_of_slot.data_ptr(), k.data_ptr(), q_pair.data_ptr(), v.data_ptr(),
        v_pair.data_ptr(), lse3.data_ptr(), None, P, E, heads, d, code, ws.data_ptr(), ws.numel(),
        stream), "attention")
    m3 = torch.empty_like(m)
    m3[pairs.by_type] = typed_rows(v_pair, pairs.by_type, msg)
    assert not torch.isfinite(lse).all()
    assert torch.equal(torch.isnan(lse), torch.isnan(lse3))
    same = ~torch.isnan(lse)
    # each within tol of the exact value
    tol = 2 * TOL_BF16 if bf16 else 2 * TOL_F32
    assert_close(lse[same].cpu().numpy(), lse3[same].cpu().numpy(), 2 * tol, "lse")
    # (a product of two or four heads spreads what is not finite over them: whole rows)
    rows = torch.isfinite(m3.float()).all(1)
    assert bool(rows.any()) and not bool(rows.all())
    assert_close(m[rows].float().cpu().numpy(), m3[rows].float().cpu().numpy(), 2 * tol, "m")


@pytest.mark.parametrize("heads,d,bf16", [(1, 64, False), (8, 16, True)])
def test_more_than_a_million_pairs(device, heads, d, bf16):
    """More tiles than the chip holds many times over, counts per relation that are no
    multiples of a tile: pass against the three launches, whole operator."""
    P, per = 1_048_613, [300_001, 17, 450_065, 298_530]
    assert sum(per) == P
    rng = np.random.default_rng(5)
    n = 460_000
    dst = [np.sort(rng.permutation(n)[:p]) for p in per]
    cnt = [rng.integers(1, 4, p) for p in per]
    dst, et = np.concatenate([np.repeat(a, c) for a, c in zip(dst, cnt)]), \
        np.repeat(np.arange(4), [c.sum() for c in cnt])
    g = prepare_graph(rng.integers(0, n, dst.size), dst, n, device=device, etype_of=et, num_etypes=4)
    pairs, dt = g.relation_pairs(), torch.bfloat16 if bf16 else torch.float32
    assert pairs.num_pairs == P
    gen = torch.Generator(device=device)
    gen.manual_seed(1)
    rand = lambda *s: torch.randn(*s, generator=gen, device=device).to(dt)
    k, q, v = (rand(n, heads * d) for _ in range(3))
    att, msg = (rand(4, heads, d, d) / d ** 0.5 for _ in range(2))
    args = (k, q, v, att, msg, None, g, 1.0 / d ** 0.5)
    assert capi.load().ga_pair_attention_preferred(P, g.num_edges, pairs.max_slots, heads, d,
                                                   capi.GA_BF16 if bf16 else capi.GA_F32)
    one = ops.relation_pair_attention(*args)
    pairs.max_slots = 257                   # a claim the pass refuses
    three = ops.relation_pair_attention(*args)
    tol = 2 * (2 * TOL_BF16 if bf16 else 2 * TOL_F32)       # each within its own of the exact value
    assert_close(one.float().cpu().numpy(), three.float().cpu().numpy(), tol, f"{heads}x{d}")


@pytest.mark.parametrize("heads,d,bf16", [(1, 64, False), (2, 32, False), (4, 16, False), (1, 64, True),
                                          (2, 64, False), (8, 16, True)])
@pytest.mark.parametrize("per", [[1], [63, 0, 65], [64, 1, 0, 129, 300] + [3] * 70])
def test_prepared_tiles(device, heads, d, bf16, per):
    """Tiles, rows and matrices prepared for the pass: the pass by itself over them gives what
    it gives without them, in by_type order, and both are within rounding of float64; more
    types than a wavefront has lanes."""
    rng = np.random.default_rng(len(per) + d)
    g, *_, n = _typed_graph(rng, per, 30, device)
    pairs, lib, T = g.relation_pairs(), capi.load(), len(per)
    tiles = pairs.tiles.cpu().numpy()
    want = [(t, lo, min(lo + 64, hi), 0) for t, (lo, hi) in enumerate(zip(
        pairs.type_pointer.tolist(), pairs.type_pointer.tolist()[1:])) for lo in range(lo, hi, 64)]
    assert [tuple(x) for x in tiles[:len(want)]] == want and (tiles[len(want):, 0] == -1).all()
    by_type = pairs.by_type
    assert torch.equal(pairs.rows[:, 0], pairs.pair_pointer[by_type])
    assert torch.equal(pairs.rows[:, 1], pairs.pair_pointer[by_type + 1])
    assert torch.equal(pairs.rows[:, 2].long(), pairs.dst_by_type)
    dt, code = (torch.bfloat16, capi.GA_BF16) if bf16 else (torch.float32, capi.GA_F32)
    rand = lambda *s: torch.from_numpy(rng.standard_normal(s, dtype=np.float32)).to(device).to(dt)
    k, q, v = (rand(n, heads * d) for _ in range(3))
    att, msg = (rand(T, heads, d, d) / d ** 0.5 for _ in range(2))
    rc, m, lse = _one_pass(g, k, q, v, att, msg)
    assert rc == capi.GA_OK
    m2, lse2 = torch.empty_like(m), torch.empty_like(lse)
    a, b = att, msg
    nbytes = lib.ga_pair_weights_bytes(T, heads, d, code)
    assert (nbytes > 0) == (not bf16 and heads * d == 64 and d >= 32)
    if nbytes:
        a, b = (torch.empty(nbytes, dtype=torch.uint8, device=device) for _ in range(2))
        scale = torch.full((T, heads), 2.0, device=device)
        capi.check(lib.ga_pair_weights(
            att.transpose(2, 3).contiguous().data_ptr(), scale.data_ptr(), capi.GA_F32, 0.5,
            msg.data_ptr(), a.data_ptr(), b.data_ptr(), T, heads, d, 0), "weights")
    run = lambda nodes: lib.ga_pair_attention_tiles(
        pairs.rows.data_ptr(), pairs.tiles.data_ptr(), T, g.in_node_indices.data_ptr(), q.data_ptr(),
        k.data_ptr(), v.data_ptr(), a.data_ptr(), b.data_ptr(), m2.data_ptr(), lse2.data_ptr(),
        pairs.num_pairs, nodes, pairs.max_slots, heads, d, code, torch.cuda.current_stream().cuda_stream)
    assert run(2 ** 31 - 1) == capi.GA_EUNSUPPORTED       # offsets past 4 GB
    capi.check(run(n), "tiles")
    if not nbytes:
        assert torch.equal(m[by_type], m2) and torch.equal(lse[by_type], lse2)
        return
    ref_m, ref_lse = _by_pair(g, k, q, v, att, msg)
    at = by_type.cpu()
    assert_close(m2.cpu().numpy(), ref_m[at].numpy(), 2 * TOL_F32, "m")
    assert_close(lse2.cpu().numpy(), ref_lse[at].numpy(), 2 * TOL_F32, "lse")
    # rows with values that are not finite: the same rows as the fp32 products give
    src, e = g.in_node_indices.long(), g.num_edges
    q[pairs.pair_dst[0].long(), 5] = float("inf")
    v[src[e - 1], 7], v[src[e // 2], :] = -float("inf"), float("nan")
    rc, m, lse = _one_pass(g, k, q, v, att, msg)
    capi.check(run(n), "tiles")
    for x, y in ((m[by_type], m2), (lse[by_type], lse2)):
        assert torch.equal(torch.isnan(x), torch.isnan(y)) and torch.equal(x == float("inf"), y == float("inf"))
        both = torch.isfinite(x)
        assert torch.equal(both, torch.isfinite(y))
        if bool(both.any()):
            assert_close(x[both].cpu().numpy(), y[both].cpu().numpy(), 4 * TOL_F32, "finite")
    assert not bool(torch.isfinite(m2).all())
