"""Projected rows kept apart (ga_gather_row_stride): the projection, the fused aggregation
and the GAT layer give what they give over rows side by side."""
import numpy as np
import pytest
import torch

from graphiler_amd import capi, layers, ops, prepare_graph


def test_rule_on_the_host():
    f = capi.load().ga_gather_row_stride
    assert f(200_000, 64, capi.GA_F32) == 96 and f(200_000, 256, capi.GA_BF16) == 320
    assert f(16_384, 64, capi.GA_F32) == 64 and f(16_385, 64, capi.GA_F32) == 96      # 4 MB
    for feat, dt in ((32, capi.GA_F32), (96, capi.GA_F32), (64, capi.GA_BF16), (100, capi.GA_F32)):
        assert f(1 << 20, feat, dt) == feat


def _graph(n, e, seed):
    rng = np.random.default_rng(seed)
    dst = rng.integers(0, n, e)
    dst[: e // 4] = 3                          # a row over many runs and workgroups
    return prepare_graph(rng.integers(0, n, e), dst, n, device="cuda:0")


@pytest.mark.gpu
@pytest.mark.parametrize("heads,dim,bf16", [(1, 64, False), (2, 32, False), (1, 128, False), (4, 16, False),
                                            (2, 64, True), (4, 64, True), (3, 64, True), (1, 128, True)])
@pytest.mark.parametrize("from_z", [0, 1])
@pytest.mark.parametrize("n,e", [(5, 0), (70, 300), (3000, 40_000)])
def test_aggregation(device, heads, dim, bf16, from_z, n, e):
    if from_z and dim == 128 and not bf16:
        pytest.skip("32 lanes to a head: not a shape of the source term from the rows")
    g, lib, feat = _graph(n, e, n + heads), capi.load(), heads * dim
    dt, code, piece = (torch.bfloat16, capi.GA_BF16, 8) if bf16 else (torch.float32, capi.GA_F32, 4)
    gen = torch.Generator(device=device).manual_seed(feat)
    z = torch.randn(n, feat, generator=gen, device=device).to(dt)
    el, er = (torch.randn(n, heads, generator=gen, device=device) for _ in range(2))
    al = torch.randn(heads, dim, generator=gen, device=device) / 8
    want = ops.gat_aggregate_from_z(al, er, z, g, 0.2, "elu") if from_z else \
        ops.gat_aggregate(el, er, z, g, 0.2, "elu")
    ws = g.workspace(lib.ga_gat_workspace_bytes(e, feat, heads))
    for pad in (0, piece, 128 // z.element_size()):
        wide = torch.full((n, feat + pad), float("nan"), dtype=dt, device=device)
        wide[:, :feat] = z
        out = torch.empty_like(z)
        call = lambda stride: lib.ga_gat_aggregate_strided(
            g.in_pointer.data_ptr(), g.in_row_of_slot.data_ptr(), g.in_node_indices.data_ptr(),
            (al if from_z else el).data_ptr(), er.data_ptr(), wide.data_ptr(), stride, out.data_ptr(),
            n, e, heads, dim, 0.2, from_z, capi.GA_ACT_ELU, code, ws.data_ptr(), ws.numel(), 0)
        assert call(feat - piece) == capi.GA_EINVAL and call(feat + 1) == capi.GA_EUNSUPPORTED
        capi.check(call(feat + pad), "strided")
        assert torch.equal(out, want)
    # float64: the logits from the stored rows, every in-edge by itself
    if e:
        zz = z.double().view(n, heads, dim)
        src = (zz * al.double()).sum(2) if from_z else el.double()
        s = torch.nn.functional.leaky_relu(src[g.COO_src] + er.double()[g.COO_dst], 0.2)
        p = torch.exp(s - s.max())
        den = torch.zeros(n, heads, dtype=torch.float64, device=device).index_add_(0, g.COO_dst, p)
        ref = torch.zeros(n, heads, dim, dtype=torch.float64, device=device).index_add_(
            0, g.COO_dst, (p / den[g.COO_dst]).unsqueeze(2) * zz[g.COO_src]).view(n, feat)
        err = (want.double() - torch.nn.functional.elu(ref)).norm() / ref.norm()
        assert float(err) < (2.0 ** -8 if bf16 else 2e-6)


@pytest.mark.gpu
@pytest.mark.parametrize("k,heads,dim,bf16", [(100, 4, 64, True), (64, 1, 128, True), (256, 2, 128, True),
                                              (602, 1, 64, False), (37, 4, 16, False), (64, 4, 32, False)])
@pytest.mark.parametrize("rows", [1, 129, 20_000])
def test_projection(device, k, heads, dim, bf16, rows):
    dt, code = (torch.bfloat16, capi.GA_BF16) if bf16 else (torch.float32, capi.GA_F32)
    gen = torch.Generator(device=device).manual_seed(k + rows)
    m = heads * dim
    x = torch.randn(rows, k, generator=gen, device=device).to(dt)
    w = (torch.randn(k, m, generator=gen, device=device) / k ** 0.5).to(dt)
    al, ar = (torch.randn(heads, dim, generator=gen, device=device) for _ in range(2))
    z, el, er = ops.linear_attn(x, w, al, ar)
    ld = m + 128 // z.element_size()
    wide = torch.full((rows, ld), 7.0, dtype=dt, device=device)
    el2, er2 = torch.empty_like(el), torch.empty_like(er)
    capi.check(capi.load().ga_project_attn_strided(
        x.data_ptr(), w.data_ptr(), al.data_ptr(), ar.data_ptr(), wide.data_ptr(), ld, el2.data_ptr(),
        er2.data_ptr(), rows, k, m, heads, code, 0), "strided")
    assert torch.equal(wide[:, :m], z) and torch.equal(el, el2) and torch.equal(er, er2)
    assert bool((wide[:, m:] == 7.0).all())


@pytest.mark.gpu
@pytest.mark.parametrize("heads,dim,bf16", [(1, 64, False), (4, 64, True), (2, 64, True), (8, 8, False)])
def test_layer(device, heads, dim, bf16, monkeypatch):
    n = 20_000 if not bf16 else 17_000        # tables above 4 MB
    g = _graph(n, 100_000, heads)
    dt = torch.bfloat16 if bf16 else torch.float32
    gen = torch.Generator(device=device).manual_seed(dim)
    h = torch.randn(n, 48, generator=gen, device=device).to(dt)
    w = (torch.randn(48, heads * dim, generator=gen, device=device) / 7).to(dt)
    a = torch.randn(2, heads, dim, generator=gen, device=device) / 4
    for limit in (1 << 40, 0):
        monkeypatch.setattr(layers, "SOURCE_TERM_TABLE_LIMIT", limit)
        apart = layers.gat_layer(g, h, w, a, heads, 0.2, activation="elu")
        with monkeypatch.context() as mp:
            mp.setattr(ops, "gat_project_and_aggregate", lambda *args: None)
            assert torch.equal(apart, layers.gat_layer(g, h, w, a, heads, 0.2, activation="elu"))


def test_shared_logits_rule_on_the_host():
    f, mb = capi.load().ga_gat_from_z_shares_logits, 1 << 20
    # rows apart; heads of other than 8 or 16 lanes
    assert f(1 << 22, 4, 64, 256 + 64, capi.GA_BF16) == 1 and f(1 << 22, 2, 64, 160, capi.GA_F32) == 1
    for heads, dim, dt in ((4, 32, capi.GA_BF16), (2, 256, capi.GA_BF16), (4, 16, capi.GA_F32),
                           (1, 128, capi.GA_F32), (1, 65, capi.GA_F32)):
        assert f(1000, heads, dim, 0, dt) == 0
    # side by side: the size of the table from which rows that share channels are left alone
    for heads, dim, dt, limit in ((4, 64, capi.GA_BF16, 768), (2, 128, capi.GA_BF16, 768),
                                  (8, 64, capi.GA_BF16, 192), (1, 64, capi.GA_F32, 64),
                                  (4, 32, capi.GA_F32, 64), (3, 32, capi.GA_F32, 640),
                                  (3, 64, capi.GA_F32, 640)):
        rows = limit * mb // (heads * dim * (4 if dt == capi.GA_F32 else 2))
        for stride in (0, heads * dim):
            assert f(rows, heads, dim, stride, dt) == 1 and f(rows + 1, heads, dim, stride, dt) == 0
    for heads in (1, 2, 3, 5):
        assert f(1 << 30, heads, 64, 0, capi.GA_BF16) == 1


@pytest.mark.gpu
@pytest.mark.parametrize("heads,dim,bf16,n", [(1, 64, False, 262_145), (2, 32, False, 262_145),
                                              (8, 64, True, 196_609)])
def test_logits_of_every_lane(device, heads, dim, bf16, n):
    """Side by side, one row past the line from which every lane forms its own logit: what the
    shared form gives over rows apart, to the rounding of a logit's sum in another order."""
    g, lib, feat, e = _graph(n, 2 * n, heads), capi.load(), heads * dim, 2 * n
    dt, code = (torch.bfloat16, capi.GA_BF16) if bf16 else (torch.float32, capi.GA_F32)
    assert not lib.ga_gat_from_z_shares_logits(n, heads, dim, 0, code)
    gen = torch.Generator(device=device).manual_seed(feat)
    z = torch.randn(n, feat, generator=gen, device=device).to(dt)
    er = torch.randn(n, heads, generator=gen, device=device)
    al = torch.randn(heads, dim, generator=gen, device=device) / 8
    got = ops.gat_aggregate_from_z(al, er, z, g, 0.2)
    wide = torch.zeros(n, feat + 128 // z.element_size(), dtype=dt, device=device)
    wide[:, :feat] = z
    out = torch.empty_like(z)
    ws = g.workspace(lib.ga_gat_workspace_bytes(e, feat, heads))
    capi.check(lib.ga_gat_aggregate_strided(
        g.in_pointer.data_ptr(), g.in_row_of_slot.data_ptr(), g.in_node_indices.data_ptr(),
        al.data_ptr(), er.data_ptr(), wide.data_ptr(), wide.shape[1], out.data_ptr(), n, e, heads, dim,
        0.2, 1, capi.GA_ACT_NONE, code, ws.data_ptr(), ws.numel(), 0), "strided")
    # logits of a few units, dim terms: weights move by less than 64 roundings of fp32; a bf16
    # result next to a border between two values goes to the other, at most 2^-7 of it away
    bound = out.double().abs() * (2.0 ** -7 if bf16 else 0) + 64 * 2.0 ** -24 * z.float().abs().max()
    assert bool(((got.double() - out.double()).abs() <= bound).all())


def _layer_inputs(device, n, k, heads, dim, dt):
    gen = torch.Generator(device=device).manual_seed(heads + dim)
    h = torch.randn(n, k, generator=gen, device=device).to(dt)
    w = (torch.randn(k, heads * dim, generator=gen, device=device) / k ** 0.5).to(dt)
    return h, w, torch.randn(2, heads, dim, generator=gen, device=device) / 4


@pytest.mark.gpu
def test_small_layers_do_not_ask_for_rows_apart(device, monkeypatch):
    """Tables that an L2 holds go straight to the two operators."""
    g = _graph(300, 2000, 1)
    want = layers.gat_layer(g, *_layer_inputs(device, 300, 48, 4, 64, torch.float32), 4, 0.2)
    def asked(*args):
        raise AssertionError("asked for rows apart")
    monkeypatch.setattr(ops, "gat_project_and_aggregate", asked)
    got = layers.gat_layer(g, *_layer_inputs(device, 300, 48, 4, 64, torch.float32), 4, 0.2)
    assert torch.equal(got, want)


@pytest.mark.gpu
def test_layer_goes_by_the_heads_of_its_vectors(device, monkeypatch):
    """``heads`` left at its default: the form of the source term follows the vectors, as the
    table of terms does."""
    n = 17_000
    g = _graph(n, 60_000, 2)
    inputs = _layer_inputs(device, n, 48, 4, 64, torch.bfloat16)
    monkeypatch.setattr(layers, "SOURCE_TERM_TABLE_LIMIT", 4 * n * 4)
    assert torch.equal(layers.gat_layer(g, *inputs, negative_slope=0.2), layers.gat_layer(g, *inputs, 4, 0.2))
