"""LayerNorm backward with as many blocks as have rows: one row, the edges of a block, of the reduction's waves and of the full
grid; the gradients of gain and shift never read a partial row that no block has written."""
import pytest
import torch

pytestmark = pytest.mark.gpu
DEV = "cuda:0"


@pytest.mark.parametrize("dtype", [torch.float32, torch.bfloat16], ids=["fp32", "bf16"])
@pytest.mark.parametrize("rows,cols", [(1, 64), (15, 128), (16, 128), (17, 128), (256, 72), (257, 512), (2040, 128), (4095, 64), (4097, 64), (9, 2304)])
def test_layernorm_bwd_row_counts(hiplib, dtype, rows, cols):
    g = torch.Generator().manual_seed(rows + cols)
    x, dy, gain = (torch.randn(*s, generator=g).to(dtype).to(DEV) for s in ((rows, cols), (rows, cols), (cols,)))
    mean, rinv = x.double().mean(1).float(), (1 / (x.double().var(1, unbiased=False) + 1e-5).sqrt()).float()
    dx, dgain, dshift = torch.empty_like(x), torch.full((cols,), 0.5, device=DEV), torch.full((cols,), -0.5, device=DEV)
    ws = torch.full((hiplib.layernorm_bwd_workspace(cols),), float("nan"), device=DEV)
    hiplib.layernorm_bwd(x, gain, mean, rinv, dy, None, dx, dgain, dshift, ws, hiplib.LN_STANDARD, 1e-5)
    xh = (x.double() - mean.double()[:, None]) * rinv.double()[:, None]
    d = dy.double() * gain.double()
    want = rinv.double()[:, None] * (d - d.mean(1, keepdim=True) - xh * (d * xh).mean(1, keepdim=True))
    # a sum of `rows` products in fp32: rows roundings of at most eps = 2^-24 each, and the few of a product
    eps = (rows + 8) * 2.0 ** -24
    assert bool(((dgain.double() - 0.5 - (dy.double() * xh).sum(0)).abs() <= eps * (1 + (dy.double() * xh).abs().sum(0))).all())
    assert bool(((dshift.double() + 0.5 - dy.double().sum(0)).abs() <= eps * (1 + dy.double().abs().sum(0))).all())
    # dx: two sums of `cols` terms; in bf16 the rounding of what is stored
    assert float((dx.double() - want).norm() / want.norm()) < (2.0 ** -8 if dtype == torch.bfloat16 else 1e-5)
