"""Linear layers as output tiles (lintile.hip): every tile form, tile edges, remainders of the contraction, every epilogue."""
import pytest
import torch
import torch.nn.functional as F

from gpu_util import DEV, rel_err

pytestmark = pytest.mark.gpu
TOL = {torch.float16: 2e-3, torch.bfloat16: 1.6e-2}


def ops():
    from pointtransformerv3_amd import ops
    return ops


def _layer(k, nout, n, dtype):
    g = torch.Generator().manual_seed(k + 3 * nout + n)
    x = torch.randn(n, k, generator=g).to(dtype)
    w = (torch.randn(nout, k, generator=g) / k ** 0.5).to(dtype)
    b = (torch.randn(nout, generator=g) * 0.5).to(dtype)
    return x, w, b


# 32 x 32 tiles: one wave's contraction, remainders of 4 waves x 1, 2, 4 steps; 64 x 64: 1, 2, 4 steps ahead; 128 x 128
FORMS = [(32, 32, 1), (32, 96, 33), (96, 32, 700), (64, 64, 31), (160, 64, 65), (224, 32, 100), (352, 32, 64), (512, 64, 17), (704, 32, 9),
         (64, 192, 5000), (192, 64, 9001), (128, 384, 4001), (384, 128, 6017), (256, 768, 2049), (512, 512, 1000), (768, 256, 3001),
         (512, 512, 6001), (1024, 128, 24_065), (2048, 512, 6100)]


@pytest.mark.parametrize("dtype", [torch.float16, torch.bfloat16])
@pytest.mark.parametrize("k,nout,n", FORMS)
def test_forms(k, nout, n, dtype):
    x, w, b = _layer(k, nout, n, dtype)
    want = F.linear(x.float(), w.float(), b.float())
    o = ops()
    if k % 128 == 0 and nout % 128 == 0:
        r = torch.randn(n, nout, generator=torch.Generator().manual_seed(1)).to(dtype)
        got = o.linear_gemm(x.to(DEV), w.to(DEV), b.to(DEV), r.to(DEV))
        assert rel_err(got, want + r.float()) < TOL[dtype]
    if k in (32, 64, 96, 128, 192, 256, 384, 512):
        got = o.linear_rows(x.to(DEV), w.to(DEV), b.to(DEV))
        assert rel_err(got, want) < TOL[dtype]
        again = o.linear_rows(x.to(DEV), w.to(DEV), b.to(DEV))
        assert torch.equal(got, again)


@pytest.mark.parametrize("dtype", [torch.float16, torch.bfloat16])
@pytest.mark.parametrize("k,nout,n", [(32, 128, 333), (64, 256, 5000), (128, 512, 8001), (256, 1024, 3000), (512, 2048, 2600), (512, 2048, 40)])
def test_gelu_with_its_input_kept_and_its_gradient(k, nout, n, dtype):
    x, w, b = _layer(k, nout, n, dtype)
    o = ops()
    pre, act = o.linear_gelu(x.to(DEV), w.to(DEV), b.to(DEV))
    want = F.linear(x.float(), w.float(), b.float())
    assert rel_err(pre, want) < TOL[dtype] and rel_err(act, F.gelu(pre.float()).cpu()) < 2 * TOL[dtype]
    z = pre.double().cpu().requires_grad_(True)
    F.gelu(z).backward(F.linear(x.double(), w.double()))
    assert rel_err(o.linear_gelu_bwd(x.to(DEV), w.to(DEV), pre), z.grad) < 2 * TOL[dtype]


@pytest.mark.parametrize("dtype", [torch.float16, torch.bfloat16])
@pytest.mark.parametrize("c,n", [(64, 1), (64, 4096), (256, 600), (512, 77), (512, 4096)])
def test_block_tail_few(c, n, dtype):
    o = ops()
    assert o.block_tail_few_pays(n, c)
    torch.manual_seed(c + n)
    proj, ln, fc1, fc2 = torch.nn.Linear(c, c), torch.nn.LayerNorm(c), torch.nn.Linear(c, 4 * c), torch.nn.Linear(4 * c, c)
    ln.weight.data.uniform_(0.5, 1.5)
    mods = [m.to(dtype).requires_grad_(False) for m in (proj, ln, fc1, fc2)]
    attn, short = torch.randn(n, c).to(dtype), torch.randn(n, c).to(dtype)
    lin = lambda m, x: F.linear(x, m.weight.float(), m.bias.float())
    s = short.float() + lin(proj, attn.float())
    want = s + lin(fc2, F.gelu(lin(fc1, F.layer_norm(s, (c,), ln.weight.float(), ln.bias.float(), ln.eps))))
    for m in mods:
        m.to(DEV)
    got = o.block_tail_few(attn.to(DEV), short.to(DEV), proj, ln, fc1, fc2)
    assert rel_err(got, want) < 2 * TOL[dtype]


@pytest.mark.parametrize("c,n", [(64, 33), (64, 2000), (256, 1), (256, 31), (256, 200), (256, 208)])
def test_block_tail_few_with_its_norm_in_front(c, n):
    """Sizes whose LayerNorm is formed by the layer behind it: one row, a last tile of one row, as many tiles as CUs."""
    test_block_tail_few(c, n, torch.float16)
    test_block_tail_few(c, n, torch.bfloat16)
