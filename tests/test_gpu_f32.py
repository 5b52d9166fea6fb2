"""The fp32 matrix-core products: Linear layers and the pair form of the convolution, at tile edges and odd widths."""
import numpy as np
import pytest
import torch

from gpu_util import DEV, rel_err, to_dev, unique_voxels
from oracle import functional as OF
from oracle import indexing as OI

pytestmark = pytest.mark.gpu


def ops():
    from pointtransformerv3_amd import ops as o
    return o


@pytest.mark.parametrize("n,k,nout", [(1, 32, 32), (63, 6, 32), (64, 16, 64), (65, 17, 65), (129, 64, 33), (1000, 130, 192),
                                      (40_000, 64, 256), (70_000, 32, 128), (20_000, 128, 512)])
@pytest.mark.parametrize("gelu,resid", [(False, False), (True, True)])
def test_linear_f32_matches_double(n, k, nout, gelu, resid):
    g = torch.Generator().manual_seed(n + k + nout)
    x, w, b = (torch.randn(*s, generator=g) for s in ((n, k), (nout, k), (nout,)))
    r = torch.randn(n, nout, generator=g) if resid else None
    want = torch.nn.functional.linear(x.double(), w.double(), b.double())
    want = torch.nn.functional.gelu(want) if gelu else want
    want = want + r.double() if resid else want
    got = ops().linear_any(x.to(DEV), w.to(DEV), b.to(DEV), gelu=gelu, resid=None if r is None else r.to(DEV))
    assert rel_err(got, want) < 2e-6


@pytest.mark.parametrize("n,k,nout", [(5, 64, 192), (2049, 512, 512)])
def test_linear_f32_halves_on_one_side(n, k, nout):
    g = torch.Generator().manual_seed(n)
    x, w, b = (torch.randn(*s, generator=g).to(DEV) for s in ((n, k), (nout, k), (nout,)))
    o = ops()
    # a half result is the float one rounded once; half rows are the same rows converted
    assert torch.equal(o.linear_f32(x, w, b, torch.float16), o.linear_f32(x, w, b).half())
    assert torch.equal(o.linear_f32(x.half(), w, b), o.linear_f32(x.half().float(), w, b))


@pytest.mark.parametrize("k", [20, 31, 32, 33, 64, 255, 256, 260])
@pytest.mark.parametrize("x_scale,w_scale", [(1.0, 1.0), (3e3, 30.0), (1e-4, 1e-6), (1e-7, 1.0), (1.0, 1e-9), (1e30, 1.0), (1.0, 400.0)])
def test_linear_f32_ranges(k, x_scale, w_scale):
    """Scales from 1e-16 to 1e30 of whole rows, next to rows far below them: every row as exact as float sums are. A sum of k products rounded k times is off by at most k 2^-24 of the sum of their sizes; half of it, and an
    eighth of it for the longer rows, holds for either way (roundings do not all point the same way)."""
    g = torch.Generator().manual_seed(k)
    x, w = torch.randn(300, k, generator=g) * x_scale, torch.randn(70, k, generator=g) * w_scale
    x[7] *= 1e-9     # one row far below the others, one of zeros
    x[8] = 0.0
    w[5] *= 1e-9
    want = x.double() @ w.double().t()
    size = x.double().abs() @ w.double().abs().t()
    got = ops().linear_f32(x.to(DEV), w.to(DEV)).cpu().double()
    bound = size * (k * 2.0 ** -24 / (8 if k >= 64 else 2)) + 1e-42
    assert ((got - want).abs() <= bound).all()


@pytest.mark.parametrize("k,half", [(6, False), (31, False), (64, False), (256, False), (8, True), (64, True), (256, True)])
@pytest.mark.parametrize("small", [1e-5, 1e-6, 1e-8, 1e-20, 1e-29, 1e-31, 1e-36])
def test_linear_f32_rows_of_mixed_magnitude(k, half, small):
    """Rows with one value of order 1 whose weights are small and the rest small, and the other way round: every value is
    held in full, so each sum is off by at most k 2^-24 of the sum of its products' sizes, k roundings, whatever else the
    row holds. A half holds 2^-24 and up: its smallest values are of 1e-5."""
    g = torch.Generator().manual_seed(k)
    x, w = torch.randn(300, k, generator=g) * (max(small, 1e-5) if half else small), torch.randn(70, k, generator=g)
    x[:, 0], w[:, 0] = 1.0 + torch.rand(300, generator=g), w[:, 0] * small
    x[100:, 1], w[35:, 2:] = torch.randn(200, generator=g), w[35:, 2:] * small
    x = x.half() if half else x
    want = x.double() @ w.double().t()
    size = x.double().abs() @ w.double().abs().t()
    got = ops().linear_f32(x.to(DEV), w.to(DEV)).cpu().double()
    bound = size * (k * 2.0 ** -24) + 1e-42
    assert ((got - want).abs() <= bound).all()


@pytest.mark.parametrize("k", [16, 64, 256])
def test_linear_f32_infinities_and_nan(k):
    g = torch.Generator().manual_seed(k)
    x, w = torch.randn(200, k, generator=g), torch.randn(70, k, generator=g)
    x[3, 5], x[10, 2], x[40, 0], w[7, 7] = float("inf"), float("nan"), 3.0e38, -float("inf")
    w[:, 0] = w[:, 0].abs() + 2.0     # 3e38 times more than two leaves the range whatever else is added
    x[40, 7] = -1.0                   # and meets no infinity of the other sign
    want = (x.double() @ w.double().t()).float()
    got = ops().linear_f32(x.to(DEV), w.to(DEV)).cpu()
    assert torch.equal(got.isnan(), want.isnan()) and torch.equal(got.isinf(), want.isinf())
    assert torch.equal(got.sign()[want.isinf()], want.sign()[want.isinf()])


@pytest.mark.parametrize("ks,cin,cout,n,extent", [(3, 32, 32, 400, 12), (3, 64, 64, 3000, 18), (3, 128, 128, 60, 5),
                                                  (3, 20, 36, 700, 10), (5, 6, 32, 900, 14), (5, 3, 5, 40, 6),
                                                  (3, 256, 256, 1500, 14)])
def test_subm_conv_pairs_f32(ks, cin, cout, n, extent):
    rng = np.random.default_rng(cin + n)
    g = torch.Generator().manual_seed(cin + n)
    grid, batch, _ = unique_voxels(rng, n, extent, 2)
    idx = np.concatenate([batch[:, None].astype(np.int32), grid], 1)
    nbr = OI.subm_kmap(idx, ks)
    feat = torch.randn(len(idx), cin, generator=g)
    w = torch.randn(cout, ks ** 3, cin, generator=g) / (ks ** 3 * cin) ** 0.5
    b = torch.randn(cout, generator=g) if ks == 3 else None
    want = OF.subm_conv(feat, nbr, w, b)
    o = ops()
    plan = o.conv_plan_direct(to_dev(idx), ks)
    got = o.subm_conv_pairs(feat.to(DEV), plan, w.to(DEV), None if b is None else b.to(DEV))
    assert rel_err(got, want) < 5e-6


@pytest.mark.parametrize("n,scale", [(200_001, 3.0), (200_001, 0.3), (4096, 1e-3), (4096, 1e3)])
def test_gelu_of_a_float_layer(n, scale):
    """x Phi(x) of a layer that hands its input through, against 64 bits: the exponential is within two ulp and takes an
    argument rounded once, the last step rounds once, so the result is off by 2^-23 of |x| at most."""
    o = ops()
    x = torch.randn(n, 1, generator=torch.Generator().manual_seed(1)) * scale
    x[:8, 0] = torch.tensor([0.0, 13.4, -13.4, 13.6, -13.6, 1e30, -1e30, -1e-30])
    got = o.linear_any(x.to(DEV), torch.ones(1, 1, device=DEV), None, gelu=True).cpu().double()
    want = x.double() * 0.5 * torch.erfc(-x.double() / 2 ** 0.5)
    assert ((got - want).abs() <= 2.0 ** -23 * x.double().abs()).all()
    odd = torch.tensor([[float("inf")], [-float("inf")], [float("nan")]], device=DEV)
    out = o.linear_any(odd, torch.ones(1, 1, device=DEV), None, gelu=True)
    assert float(out[0]) == float("inf") and torch.isnan(out[1:]).all()
