"""The fused aggregation's bf16 build for rows that leave lanes of their group idle and for
short lists, on both sides of its lines, against float64."""
import numpy as np
import pytest
import torch

from graphiler_amd import ops, prepare_graph

pytestmark = pytest.mark.gpu


# lanes of 8 features: 24 of 32 and 40 of 64 idle some, 32 and 64 none; a second feature tile
@pytest.mark.parametrize("heads,dim,n,e", [(3, 64, 70, 300), (5, 64, 500, 9000), (9, 64, 300, 3000),
                                           (2, 24, 300, 3000), (4, 64, 500, 9000), (8, 64, 70, 300),
                                           (4, 64, 3000, (1 << 20) - 1), (4, 64, 3000, 1 << 20)])
@pytest.mark.parametrize("activation", [None, "relu", "elu"])
def test_against_float64(device, heads, dim, n, e, activation):
    rng = np.random.default_rng(e + heads)
    dst = rng.integers(0, n - 1, e)                # the last row has no edge
    dst[: min(e // 4, 3000)] = 3                   # a row over many runs
    g = prepare_graph(rng.integers(0, n, e), dst, n, device=device)
    gen = torch.Generator(device=device).manual_seed(e)
    z = torch.randn(n, heads * dim, generator=gen, device=device).bfloat16()
    z[5, :8] = torch.tensor([float("inf"), -float("inf"), float("nan"), 0.0, -0.0, 1e30, 1e-40, 1.0])
    el, er = (torch.randn(n, heads, generator=gen, device=device) for _ in range(2))
    got = ops.gat_aggregate(el, er, z, g, 0.2, activation).double()
    zz = z.double().view(n, heads, dim)
    s = torch.nn.functional.leaky_relu(el.double()[g.COO_src] + er.double()[g.COO_dst], 0.2)
    p = torch.exp(s)
    den = torch.zeros(n, heads, dtype=torch.float64, device=device).index_add_(0, g.COO_dst, p)
    ref = torch.zeros(n, heads, dim, dtype=torch.float64, device=device)
    step = max(1, (1 << 26) // (heads * dim))
    for lo in range(0, e, step):
        at = slice(lo, min(lo + step, e))
        w = p[at] / den[g.COO_dst[at]]
        ref.index_add_(0, g.COO_dst[at], w.unsqueeze(2) * zz[g.COO_src[at]])
    ref = ref.view(n, heads * dim)
    if activation:
        ref = getattr(torch.nn.functional, activation)(ref)
    finite = torch.isfinite(ref)
    assert torch.equal(torch.isnan(ref), torch.isnan(got))
    assert torch.equal(torch.isinf(ref), torch.isinf(got) & ~torch.isnan(ref))
    # rounded to bf16 once (2^-9 of the value), weights and sums in fp32
    size = torch.where(torch.isfinite(zz), zz.abs(), 0.0).view(n, -1).max(0).values
    err = torch.where(finite, (got - ref).abs(), 0.0)
    assert bool((err <= torch.where(finite, ref.abs(), 0.0) * 2.0 ** -8 + size * 2.0 ** -17).all())
    assert bool((got[n - 1] == 0).all())
