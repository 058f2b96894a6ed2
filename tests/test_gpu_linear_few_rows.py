"""The projection in tiles of 16 rows (ga_linear_attn on small grids and few columns): edges of
its tiles, k slices and column blocks against float64, the attention terms and the row factor."""
import numpy as np
import pytest
import torch

from graphiler_amd import ops
from helpers import TOL_F32, assert_close

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("rows", [1, 15, 16, 17, 4097])
@pytest.mark.parametrize("k", [1, 7, 31, 32, 33, 256, 259, 545])
@pytest.mark.parametrize("m", [1, 16, 17, 32, 33, 64])
def test_plain(device, rows, k, m):
    """k up to 17 slices: four and eight wavefronts with none, one, two and three each."""
    gen = torch.Generator(device=device).manual_seed(rows + 100 * k + m)
    x = torch.randn(rows, k, device=device, generator=gen)
    w = torch.randn(k, m, device=device, generator=gen)
    s = torch.rand(rows, device=device, generator=gen)
    got = ops.linear(x, w)
    want, size = x.double() @ w.double(), x.double().abs() @ w.double().abs()
    assert_close(got.cpu().numpy(), want.cpu().numpy(), TOL_F32, "z", mag=size.cpu().numpy())
    assert torch.equal(ops.linear(x, w, row_scale=s), got * s[:, None])
    # a row that is not finite stays alone, and so does a column of the weights
    x[rows // 2, k - 1] = float("inf")
    bad = torch.isfinite(ops.linear(x, w)).all(1)
    assert not bad[rows // 2] and bad.sum() == rows - 1
    x[rows // 2, k - 1] = 1.0
    w[0, m - 1] = float("nan")
    cols = torch.isfinite(ops.linear(x, w)).all(0)
    assert not cols[m - 1] and cols[:m - 1].all()


@pytest.mark.parametrize("rows,k", [(1, 1), (17, 33), (2000, 64), (4113, 545), (16383, 130), (16383, 512)])
@pytest.mark.parametrize("m", [1, 16, 33, 64])
def test_infinities_products_that_overflow_and_small_operands(device, rows, k, m):
    """What a product of torch's below LINEAR_MIN_ROWS gives: infinities with their signs, the sign of
    a product that overflows, and operands far below 1 with all their bits."""
    gen = torch.Generator(device=device).manual_seed(rows + k + m)
    x = torch.randn(rows, k, device=device, generator=gen)
    w = torch.randn(k, m, device=device, generator=gen)
    x[0, k - 1], x[rows // 2, 0], x[rows // 3, k // 2] = float("inf"), float("-inf"), float("nan")
    w[k // 3, m // 2] = float("inf")
    got, want = ops.linear(x, w), (x.double() @ w.double()).float()
    assert torch.equal(torch.isnan(got), torch.isnan(want))
    inf = torch.isinf(want)
    assert torch.equal(got[inf], want[inf])
    # one product that overflows a sum, next to products of any sign
    x, w = torch.randn_like(x), torch.randn_like(w) / 64
    x[rows - 1], w[0, m - 1] = 0.0, -3e38
    x[rows - 1, 0], x[rows - 1, k // 2] = 3e38, 3e38
    got, want = ops.linear(x, w)[rows - 1], (x[rows - 1].double() @ w.double()).float()
    assert got[m - 1] == -float("inf") and not torch.isnan(got).any()
    assert torch.equal(torch.isinf(got), torch.isinf(want))
    # 2^-122 has all the bits of a float; the result's last one is 2^-149
    x = torch.randn(rows, k, device=device, generator=gen) * 2.0 ** -122
    w = torch.randn(k, m, device=device, generator=gen)
    want, size = x.double() @ w.double(), x.double().abs() @ w.double().abs()
    got = ops.linear(x, w).double()
    assert ((got - want).abs() <= (k + 8) * 2.0 ** -24 * size + k * 2.0 ** -149).all()


def test_a_single_product_is_rounded_once(device):
    """Rows with one value that is not zero (bag-of-words features)."""
    gen = torch.Generator(device=device).manual_seed(3)
    x, w = torch.zeros(3000, 300, device=device), torch.randn(300, 64, device=device, generator=gen)
    at = torch.randint(0, 300, (3000,), device=device, generator=gen)
    v = torch.randn(3000, device=device, generator=gen)
    x[torch.arange(3000, device=device), at] = v
    assert torch.equal(ops.linear(x, w), v[:, None] * w[at])


@pytest.mark.parametrize("rows,k", [(1, 5), (17, 64), (4096, 130), (4113, 300)])
@pytest.mark.parametrize("heads,dim", [(1, 16), (1, 32), (2, 16), (1, 64), (2, 32), (4, 16), (3, 16), (2, 64), (8, 16)])
def test_attention_terms(device, rows, k, heads, dim):
    rng = np.random.default_rng(rows + k + heads)
    x = rng.standard_normal((rows, k)).astype(np.float32)
    w = rng.standard_normal((k, heads * dim)).astype(np.float32) / np.float32(np.sqrt(k))
    a = rng.standard_normal((2, heads, dim)).astype(np.float32)
    dev = [torch.from_numpy(t).to(device) for t in (x, w, a[0], a[1])]
    z, el, er = ops.linear_attn(*dev)
    zr = (x.astype(np.float64) @ w).reshape(rows, heads, dim)
    zm = (np.abs(x).astype(np.float64) @ np.abs(w)).reshape(rows, heads, dim)
    assert_close(z.cpu().numpy(), zr.reshape(rows, -1), TOL_F32, "z", mag=zm.reshape(rows, -1))
    for got, v in ((el, a[0]), (er, a[1])):
        assert_close(got.cpu().numpy(), (zr * v).sum(2), TOL_F32, "terms", mag=(zm * np.abs(v)).sum(2))
    assert torch.equal(ops.linear_attn(*dev[:2]), z)


@pytest.mark.parametrize("rows,k,m", [(20_001, 33, 64), (40_000, 37, 17), (33_000, 45, 130), (20_480, 1433, 64),
                                      (150_001, 1, 5), (151_000, 127, 16), (40_000, 31, 33)])
def test_rows_of_an_odd_number_of_values(device, rows, k, m):
    """Grids of 128-row workgroups whose rows only four-byte accesses tile: whole and broken last
    slices, the last rows of x, columns beyond a pass, against float64."""
    gen = torch.Generator(device=device).manual_seed(rows + k + m)
    x = torch.randn(rows, k, device=device, generator=gen)
    w = torch.randn(k, m, device=device, generator=gen)
    want, size = x.double() @ w.double(), x.double().abs() @ w.double().abs()
    z = ops.linear_attn(x, w)
    assert_close(z.cpu().numpy(), want.cpu().numpy(), TOL_F32, "z", mag=size.cpu().numpy())
    x[rows - 1, k - 1] = float("nan")
    fin = torch.isfinite(ops.linear_attn(x, w)).all(1)
    assert fin[:-1].all() and not fin[-1]
    if m in (64, 16):
        a = torch.randn(2, 1, m, device=device, generator=gen)
        _, el, er = ops.linear_attn(x[:-1].contiguous(), w, a[0], a[1])
        for got, v in ((el, a[0]), (er, a[1])):
            assert_close(got.cpu().numpy(), (want[:-1] @ v.double().T).cpu().numpy(), TOL_F32, "terms",
                         mag=(size[:-1] @ v.double().abs().T).cpu().numpy())


def test_what_torch_does_with_a_product_is_kept(device):
    """Few rows are a product of torch's where it has more to do than multiply."""
    import torch.autograd.forward_ad as fwd
    x, w = torch.randn(500, 40, device=device), torch.randn(40, 24, device=device)
    s = torch.rand(500, 2, device=device)
    want = x @ w
    # fp32 products of 40 values: 40 roundings of 2^-24 each against |x| |w|
    near = lambda got, ref: bool(((got - ref).abs() <= 80 * 2 ** -24 * (x.abs() @ w.abs())).all())
    assert not ops.linear(x, w).requires_grad and near(ops.linear(x, w), want)
    p = torch.nn.Parameter(w)
    ops.linear(x, p, s[:, 1:].contiguous()).sum().backward()
    assert torch.allclose(p.grad, x.t() @ s[:, 1:].expand(-1, 24), rtol=1e-4, atol=1e-3)
    with torch.no_grad():
        assert near(ops.linear(x, p), want)
    assert torch.equal(ops.linear(x, w, s[:, 1]), want * s[:, 1:])              # a strided factor
    assert torch.allclose(torch.vmap(lambda a: ops.linear(a, w))(x[None].expand(3, -1, -1))[2], want, atol=1e-4)
    with fwd.dual_level():
        assert fwd.unpack_dual(ops.linear(fwd.make_dual(x, torch.ones_like(x)), w)).tangent is not None
    with torch.autocast("cuda", dtype=torch.bfloat16):
        assert ops.linear(x, w).dtype == torch.bfloat16
    traced = torch.jit.trace(lambda a: ops.linear(a, w), (x,), check_trace=False)
    assert torch.allclose(traced(2 * x), 2 * want, atol=1e-4)
    with pytest.raises(RuntimeError):
        ops.linear(x, w[:39].contiguous())
    with pytest.raises(RuntimeError):
        ops.linear(x, w.cpu())


def test_a_product_of_another_device_is_torchs(device, monkeypatch):
    """Kernels are launched on the current device; torch multiplies on that of its operands."""
    x, w = torch.randn(500, 40, device=device), torch.randn(40, 24, device=device)
    launched = []
    monkeypatch.setattr(ops, "linear_attn", lambda *a: launched.append(a))
    ops.linear(x, w)
    assert len(launched) == 1
    monkeypatch.setattr(torch.cuda, "current_device", lambda: x.get_device() + 1)
    assert torch.equal(ops.linear(x, w), torch.mm(x, w)) and len(launched) == 1
