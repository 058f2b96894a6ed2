"""Pair attention over tables that 32-bit offsets do not reach: the pass over the pair columns,
not the three launches."""
import numpy as np
import pytest
import torch

from graphiler_amd import capi, ops, prepare_graph, torch_boundary
from helpers import TOL_BF16, TOL_F32, assert_close


def test_rule_on_the_host():
    fit = capi.load().ga_pair_tiles_fit
    for heads, d, dt, size in ((1, 64, capi.GA_F32, 256), (8, 16, capi.GA_BF16, 256), (2, 64, capi.GA_F32, 512)):
        assert fit((2 ** 32 - 1) // size, heads, d, dt) == 1 and fit(2 ** 32 // size, heads, d, dt) == 0
    assert fit(2 ** 31, 1, 8, capi.GA_BF16) == 0 and fit(-1, 1, 64, capi.GA_F32) == 0


def _calls(monkeypatch, *names):
    lib, seen = capi.load(), []
    for name in names:
        plain = getattr(lib, name)
        monkeypatch.setattr(lib, name, lambda *a, name=name, plain=plain: (seen.append(name), plain(*a))[1])
    return seen


NAMES = ("ga_pair_attention", "ga_pair_attention_tiles", "ga_pair_weights", "ga_dot_attention_sum")


@pytest.mark.gpu
@pytest.mark.parametrize("heads,d,bf16", [(1, 64, False), (2, 32, False), (8, 16, True), (2, 64, False)])
def test_the_pass_over_pair_columns(device, heads, d, bf16, monkeypatch):
    rng = np.random.default_rng(d)
    n, types, per = 3000, 5, 4
    dst = np.tile(np.repeat(np.arange(n), per), types)
    et = np.repeat(np.arange(types), n * per)
    g = prepare_graph(rng.integers(0, n, dst.size), dst, n, device=device, etype_of=et, num_etypes=types)
    dt = torch.bfloat16 if bf16 else torch.float32
    rand = lambda *s: torch.from_numpy(rng.standard_normal(s, dtype=np.float32)).to(device).to(dt)
    k, q, v = (rand(n, heads * d) for _ in range(3))
    att, msg = (rand(types, heads, d, d) / d ** 0.5 for _ in range(2))
    scale = rand(types, heads).abs()
    call = lambda: ops.relation_pair_attention(k, q, v, att, msg, scale, g, factor=d ** -0.5)
    want = call()
    monkeypatch.setattr(capi.load(), "ga_pair_tiles_fit", lambda *a: 0)
    seen = _calls(monkeypatch, *NAMES)
    got = call()
    assert seen == ["ga_pair_attention"]
    tol = 2 * (2 * TOL_BF16 if bf16 else 2 * TOL_F32)       # each within its own of the exact value
    assert_close(got.float().cpu().numpy(), want.float().cpu().numpy(), tol, f"{heads}x{d}")


@pytest.mark.gpu
def test_tables_of_more_than_4_gb(device, monkeypatch):
    """Sources and destinations past the 2^32-th byte of their tables."""
    rng = np.random.default_rng(1)
    n, types, pairs, per = 2 ** 24 + 1000, 3, 4000, 4
    who = np.sort(np.concatenate([rng.integers(0, n, pairs - 500), np.arange(n - 500, n)]))
    who = np.unique(who)
    dst = np.tile(np.repeat(who, per), types)
    src = rng.integers(0, n, dst.size)
    src[::3] = n - 1 - rng.integers(0, 900, src[::3].size)
    et = np.repeat(np.arange(types), who.size * per)
    g = prepare_graph(src, dst, n, device=device, etype_of=et, num_etypes=types)
    gen = torch.Generator(device=device).manual_seed(1)
    k, q, v = (torch.randn(n, 64, generator=gen, device=device) for _ in range(3))
    assert k.numel() * 4 > 2 ** 32
    att, msg = (torch.randn(types, 1, 64, 64, generator=gen, device=device) / 8 for _ in range(2))
    seen = _calls(monkeypatch, *NAMES)
    got = ops.relation_pair_attention(k, q, v, att, msg, None, g, factor=0.125)
    assert seen == ["ga_pair_attention"]
    torch_boundary.load()
    same = torch.ops.my_ops.relation_pair_attention(k, q, v, att, msg, None, 8.0,
                                                    torch_boundary.script_graph(g))
    at = torch.from_numpy(who).to(device)
    assert torch.equal(got[at], same[at])
    s, r, t = (torch.from_numpy(x).to(device) for x in (src, dst, et))
    ke, ve = torch.empty(2, s.numel(), 64, dtype=torch.float64, device=device)
    for i in range(types):
        ke[t == i] = k[s[t == i]].double() @ att[i, 0].double()
        ve[t == i] = v[s[t == i]].double() @ msg[i, 0].double()
    row = torch.searchsorted(at, r)
    p = torch.exp((ke * q[r].double()).sum(1) * 0.125)
    den = torch.zeros(at.numel(), dtype=torch.float64, device=device).index_add_(0, row, p)
    ref = torch.zeros(at.numel(), 64, dtype=torch.float64, device=device).index_add_(
        0, row, (p / den[row]).unsqueeze(1) * ve)
    assert_close(got[at].cpu().numpy(), ref.cpu().numpy(), 2 * TOL_F32, "rows with edges")
