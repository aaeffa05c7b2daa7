"""BatchNorm forward from strip statistics: channels that end inside a block's 32 or inside the pair of such that shares lines, grids
that blocks fill up, one strip, a ragged last strip, the most rows it takes."""
import pytest
import torch

pytestmark = pytest.mark.gpu
DEV = "cuda:0"


@pytest.mark.parametrize("rows,cols", [(2, 8), (32, 32), (33, 40), (511, 64), (513, 72), (900, 96), (1000, 264), (8192, 128), (8161, 8), (300, 2088), (6272, 1024)])
def test_batchnorm_from_strips(hiplib, rows, cols):
    g = torch.Generator().manual_seed(rows + cols)
    rand = lambda *s: torch.randn(*s, generator=g).bfloat16().to(DEV)
    x, res, gamma, beta = rand(rows, cols), rand(rows, cols), rand(cols), rand(cols)
    strips = torch.zeros((rows + 31) // 32, 3, cols, device=DEV)
    for q, b in enumerate(x.float().split(32)):
        strips[q] = torch.stack([b[0], (b - b[0]).sum(0), ((b - b[0]) ** 2).sum(0)])
    y = torch.full_like(x, float("nan"))
    mean, rstd, rm, rv = (torch.full((cols,), v, device=DEV) for v in (float("nan"), float("nan"), 0.5, 2.0))
    hiplib.batchnorm_fwd(x, gamma, beta, res, y, mean, rstd, rm, rv, None, 1e-5, 0.1, True, strip_stats=strips.reshape(-1))
    xd = x.double()
    mu, var = xd.mean(0), xd.var(0, unbiased=False)
    # sums over at most 8192 rows in 16 shares of 16 strips of 32: a few dozen roundings of eps = 2^-24 on terms of order one
    assert float((mean.double() - mu).abs().max()) < 64 * 2.0 ** -24 * (1 + float(xd.abs().max()))
    assert float((rstd.double() * (var + 1e-5).sqrt() - 1).abs().max()) < 256 * 2.0 ** -24
    assert torch.allclose(rm.double(), 0.45 + 0.1 * mu, atol=1e-5) and torch.allclose(rv.double(), 1.8 + 0.1 * xd.var(0), atol=1e-4)
    # what is stored: a rounding to bf16 of a value whose own error is some fp32 roundings of its terms
    want = ((xd - mu) / (var + 1e-5).sqrt() * gamma.double() + beta.double() + res.double()).clamp(min=0)
    assert bool(((y.double() - want).abs() <= 2.0 ** -8 * want.abs() + 1e-4).all())
