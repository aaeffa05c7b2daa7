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


# The parameter gradients left as sums per block and added up beside weight gradients: in every kernel that a group may take (eight
# and four waves, 128x128 tiles free and in lock step; fp32 tiles and waves), one problem at a time where it may take none, and by
# themselves.  Two LayerNorms, columns that are no multiple of a block's 64; the same bits as one call after the other, and the
# weight gradients' too.
@pytest.mark.parametrize("dtype,rows,cols,ffn", [(torch.bfloat16, 5, 72, 64), (torch.bfloat16, 128, 128, 512), (torch.bfloat16, 300, 512, 2048),
                                                 (torch.bfloat16, 1050, 520, 2048), (torch.bfloat16, 700, 1600, 6400), (torch.bfloat16, 8192, 1024, 4096),
                                                 (torch.bfloat16, 64, 1032, 40), (torch.float32, 128, 128, 512), (torch.float32, 300, 512, 2048),
                                                 (torch.float32, 36, 68, 4)])
def test_parameter_gradients_beside_weight_gradients(hiplib, dtype, rows, cols, ffn):
    g = torch.Generator().manual_seed(rows + cols)
    rand = lambda *s: torch.randn(*s, generator=g).to(dtype).to(DEV)
    x, dy, res, gain = rand(rows, cols), rand(rows, cols), rand(rows, cols), rand(cols)
    mean, rinv = x.float().mean(1), 1 / (x.float().var(1, unbiased=False) + 1e-5).sqrt()
    act = rand(rows, ffn)
    outs = []
    for how in ("one by one", "beside", "by themselves"):
        dx = [torch.empty_like(x) for _ in range(2)]
        vec = [torch.full((cols,), 0.5, device=DEV) for _ in range(4)]
        ws = [torch.full((hiplib.layernorm_bwd_workspace(cols),), float("nan"), device=DEV) for _ in range(2)]
        W = [torch.ones(cols, cols, device=DEV), torch.ones(ffn, cols, device=DEV), torch.ones(cols, ffn, device=DEV)]
        descs = [hiplib.gemm_desc(hiplib.TN, a, b, c, accumulate=True) for a, b, c in ((dy, x, W[0]), (act, x, W[1]), (dy, act, W[2]))]
        sums = []
        for i, d in enumerate((dy, res)):
            args = (x, gain, mean, rinv, d, res if i == 0 else None, dx[i], vec[2 * i], vec[2 * i + 1], ws[i], hiplib.LN_STANDARD, 1e-5)
            if how == "one by one":
                hiplib.layernorm_bwd(*args)
            else:
                sums.append(hiplib.layernorm_bwd_rows(*args))
        if how == "by themselves":
            hiplib.partial_sums(sums)
        hiplib.gemm_grouped(descs, sums=sums if how == "beside" else ())
        outs.append(dx + vec + W)
    assert all(torch.equal(a, b) for other in outs[1:] for a, b in zip(outs[0], other))
    with pytest.raises(hiplib.HipKernelError):
        hiplib.gemm_grouped(descs, sums=sums * 3)      # more than a launch takes


# The gradient behind a dropout, written beside the one in front of it: the same bits as the dropout of what is stored, and dx and the
# parameter gradients as without; every width of the kernel, with and without a residual; a probability too small to drop anything.
@pytest.mark.parametrize("dtype", [torch.float32, torch.bfloat16], ids=["fp32", "bf16"])
@pytest.mark.parametrize("rows,cols,p", [(1, 64, 0.1), (37, 72, 0.5), (4097, 512, 0.1), (300, 1032, 0.1), (50, 2304, 0.3), (21, 4104, 0.1), (40, 128, 1e-7)])
def test_gradient_behind_a_dropout(hiplib, dtype, rows, cols, p):
    if dtype == torch.float32 and cols > 4096:
        cols = 4096
    g = torch.Generator().manual_seed(rows + cols)
    x, dy, res, gain = (torch.randn(*s, generator=g).to(dtype).to(DEV) for s in ((rows, cols), (rows, cols), (rows, cols), (cols,)))
    mean, rinv = x.float().mean(1), 1 / (x.float().var(1, unbiased=False) + 1e-5).sqrt()
    for dres in (None, res):
        outs = []
        for together in (False, True):
            dx, dropped = torch.empty_like(x), torch.full_like(x, float("nan"))
            vec = [torch.zeros(cols, device=DEV) for _ in range(2)]
            ws = torch.full((hiplib.layernorm_bwd_workspace(cols),), float("nan"), device=DEV)
            kw = dict(dropped=dropped, dropout=(p, (11, 23))) if together else {}
            hiplib.partial_sums([hiplib.layernorm_bwd_rows(x, gain, mean, rinv, dy, dres, dx, *vec, ws, hiplib.LN_STANDARD, 1e-5, **kw)])
            if not together:
                hiplib.dropout_apply(dx, dropped, p, (11, 23))
            outs.append([dx, dropped, *vec])
        assert all(torch.equal(a, b) for a, b in zip(*outs))


# Two LayerNorms whose parameters are one (and a third beside them): sums that meet in the same memory, or in a part of it, are added
# one after the other; the bits of calls one by one, in a launch of their own and beside weight gradients.
@pytest.mark.parametrize("dtype", [torch.float32, torch.bfloat16], ids=["fp32", "bf16"])
@pytest.mark.parametrize("shift", [0, 64])
def test_sums_into_the_same_gradients(hiplib, dtype, shift):
    rows, cols = 300, 136
    g = torch.Generator().manual_seed(shift)
    rand = lambda *s: torch.randn(*s, generator=g).to(dtype).to(DEV)
    x, dys, gain = rand(rows, cols), [rand(rows, cols) for _ in range(3)], rand(cols)
    mean, rinv = x.float().mean(1), 1 / (x.float().var(1, unbiased=False) + 1e-5).sqrt()
    outs = []
    for how in ("one by one", "by themselves", "beside"):
        store, W = torch.full((4, 256), 0.5, device=DEV), [torch.ones(cols, cols, device=DEV) for _ in range(2)]
        into = [(store[0, :cols], store[1, :cols]), (store[1, shift:shift + cols], store[0, shift:shift + cols]), (store[2, :cols], store[3, :cols])]
        sums = []
        for dy, (dgain, dshift) in zip(dys, into):
            ws = torch.full((hiplib.layernorm_bwd_workspace(cols),), float("nan"), device=DEV)
            args = (x, gain, mean, rinv, dy, None, torch.empty_like(x), dgain, dshift, ws, hiplib.LN_STANDARD, 1e-5)
            if how == "one by one":
                hiplib.layernorm_bwd(*args)
            else:
                sums.append((hiplib.layernorm_bwd_rows(*args), ws))
        if how == "by themselves":
            hiplib.partial_sums([s for s, _ in sums])
        descs = [hiplib.gemm_desc(hiplib.TN, dy, x, w, accumulate=True) for dy, w in zip(dys, W)]
        hiplib.gemm_grouped(descs, sums=[s for s, _ in sums] if how == "beside" else ())
        outs.append([store] + W)
    assert all(torch.equal(a, b) for other in outs[1:] for a, b in zip(outs[0], other))
