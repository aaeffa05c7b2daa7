"""Products whose epilogue works on the accumulators in registers, and whose operands are reached by 32-bit offsets from a base
per tile: rows and columns off the tile, every epilogue kind, results in fp32, leading dimensions on either side of the limit."""
import itertools

import pytest
import torch

pytestmark = pytest.mark.gpu
DEV = "cuda:0"


def rand(*shape, seed, scale=1.0):
    g = torch.Generator(device=DEV).manual_seed(seed)
    return (torch.randn(*shape, generator=g, device=DEV) * scale).bfloat16()


def framed(M, N, dtype=torch.bfloat16, guard=True):
    wide = torch.full((M + guard, N + 8 * guard), 7.0, dtype=dtype, device=DEV)
    return wide, wide[:M, :N]


# tile the shape takes; a row or column group of a tile alone, whole tiles, some short of whole
@pytest.mark.parametrize("tile,M,N,K", [("64x64k64s4", 1, 8, 64), ("64x64k64s4", 33, 40, 128), ("64x64k64s4", 1050, 512, 192), ("k64s3", 2300, 1040, 448),
                                        ("128x128k64s3", 3301, 1032, 512), ("256x128k64s3", 8100, 1000, 512), ("256x128k64s3", 8192, 1024, 512)])
@pytest.mark.parametrize("layout", ["nt", "nn"])
def test_register_epilogue(hiplib, layout, tile, M, N, K):
    for guard in (True, False):     # outputs inside wider buffers, whose rest stays as it is, or contiguous ones
        every_kind(hiplib, layout, tile, M, N, K, guard)


# ... the half tiles and 128x128 by their whole names: which of them a shape takes depends on the contraction, too
@pytest.mark.parametrize("variant,M,N,K", [("bf16_nt_dma128x64k64s3", 2041, 776, 448), ("bf16_nt_dma128x64k64s3", 627, 3264, 832), ("bf16_nn_dma64x128k64s3", 2041, 776, 448),
                                           ("bf16_nn_dma64x128k64s3", 2041, 776, 1600), ("bf16_nt_dma64x128k64s3", 2041, 776, 832), ("bf16_nt_dma64x128k64s5", 2041, 776, 1600),
                                           ("bf16_nt_dma128x128k64s3", 2300, 1040, 448), ("bf16_nn_dma128x128k64s3", 2300, 1040, 448),
                                           ("bf16_nn_short_dma256x128k64s3", 8100, 1000, 192),
                                           ("bf16_nn_whole_dma256x128k64s3", 8100, 1000, 320), ("bf16_nt_whole_dma256x128k64s3", 8100, 1000, 320), ("bf16_nt_dma256x128k64s3", 8100, 1000, 768)])
def test_register_epilogue_of_half_tiles(hiplib, variant, M, N, K):
    for guard in (True, False):
        every_kind(hiplib, variant[5:7], variant, M, N, K, guard)


def every_kind(hiplib, layout, tile, M, N, K, guard):
    lay = hiplib.NT if layout == "nt" else hiplib.NN
    A, B = rand(M, K, seed=1), rand(*((N, K) if layout == "nt" else (K, N)), seed=2, scale=0.2)
    bias, X, R = rand(N, seed=3), rand(M, N, seed=4), rand(M, N, seed=5)
    (wide, C), (wide2, D) = (framed(M, N, guard=guard) for _ in range(2))
    assert hiplib.gemm_variant(hiplib.gemm_desc(lay, A, B, C)).endswith(tile)
    a, b = A.double(), (B.double().t() if layout == "nt" else B.double()).contiguous()
    prod, slack = a @ b, K * 2.0 ** -24 * (a.abs() @ b.abs())
    x, r, u = X.double(), R.double(), prod + bias.double()

    # the sums' K eps sum |a b|, a few roundings of what is added in fp32, and half an ulp of the bf16 result (at most 2^-8)
    def near(got, want, scale=1.0):
        s = scale * (slack + 2.0 ** -22 * (prod.abs() + 8.0))
        assert ((got.double() - want).abs() <= 2.0 ** -8 * want.abs() + 1.01 * s).all()
        assert (wide[M:] == 7).all() and (wide[:, N:] == 7).all() and (wide2[M:] == 7).all() and (wide2[:, N:] == 7).all()

    hiplib.gemm(lay, A, B, C)
    near(C, prod)
    hiplib.gemm(lay, A, B, C, bias=bias, alpha=0.5)
    near(C, 0.5 * prod + bias.double())
    hiplib.gemm(lay, A, B, C, bias=bias, epilogue=hiplib.EPI_RESIDUAL, resid=R)
    near(C, u + r)
    hiplib.gemm(lay, A, B, C, epilogue=hiplib.EPI_MUL, aux_in=X)
    near(C, prod * x, scale=x.abs())
    hiplib.gemm(lay, A, B, C, epilogue=hiplib.EPI_MUL_POS, aux_in=X, resid=R)
    near(C, torch.where(x > 0, prod + r, 0.0))
    hiplib.gemm(lay, A, B, C, epilogue=hiplib.EPI_DACT, act=hiplib.ACT_RELU, aux_in=X)
    near(C, torch.where(x > 0, prod, 0.0))
    hiplib.gemm(lay, A, B, C, bias=bias, epilogue=hiplib.EPI_ACT, act=hiplib.ACT_RELU, aux_out=D)
    near(D, u)
    near(C, u.clamp_min(0))
    hiplib.gemm(lay, A, B, C, bias=bias, epilogue=hiplib.EPI_ACT_DACT, act=hiplib.ACT_GELU_TANH, aux_out=D)
    g = u.clone().requires_grad_()
    y = torch.nn.functional.gelu(g, approximate="tanh")
    dy, = torch.autograd.grad(y.sum(), g)
    near(C, y.detach(), scale=2.0)      # |gelu'| and |gelu''| stay below 1.2
    near(D, dy.double(), scale=2.0)
    F0 = torch.randn(M, N, generator=torch.Generator(device=DEV).manual_seed(6), device=DEV)
    wide3, F = framed(M, N, torch.float32, guard)
    F.copy_(F0)
    hiplib.gemm(lay, A, B, F, accumulate=True)
    assert ((F.double() - prod - F0.double()).abs() <= slack + 2.0 ** -23 * (prod.abs() + F0.double().abs() + 1.0)).all()
    assert (wide3[M:] == 7).all() and (wide3[:, N:] == 7).all()


def apart(t, step):
    """The same matrix, its rows ``step`` elements apart."""
    far = torch.empty(t.shape[0] * step, dtype=t.dtype, device=DEV).view(t.shape[0], step)[:, : t.shape[1]]
    return far.copy_(t)


@pytest.mark.parametrize("layout", ["nt", "nn"])
def test_rows_far_apart(hiplib, layout):
    M, N, K, ld = 130, 136, 128, 1 << 22
    lay = hiplib.NT if layout == "nt" else hiplib.NN
    a, b = rand(M, K, seed=1), rand(*((N, K) if layout == "nt" else (K, N)), seed=2)
    for far, step in itertools.product("AB", (ld, ld - 8)):
        A, B = (apart(a, step), b) if far == "A" else (a, apart(b, step))
        C, D = (torch.empty(M, N, dtype=torch.bfloat16, device=DEV) for _ in range(2))
        variant = hiplib.gemm_variant(hiplib.gemm_desc(lay, A, B, C))
        assert variant.endswith("128x128k64r") == (step == ld)
        hiplib.gemm(lay, A, B, C)
        hiplib.gemm(lay, a, b, D)
        assert torch.equal(C, D)         # the kernels add up a contraction in one order
        hiplib.gemm_grouped([hiplib.gemm_desc(lay, A, B, C), hiplib.gemm_desc(lay, A, B, D)])
        assert torch.equal(C, D)


@pytest.mark.parametrize("far", ["A", "B"])
@pytest.mark.parametrize("step", [1 << 22, (1 << 22) - 8])
def test_column_statistics_of_rows_far_apart(hiplib, far, step):
    """The kernels that leave column sums, forward (of a convolution's output) and backward (of a normalisation's gradient): as from contiguous
    operands, whose tiles they may not share; a strip's rows are added in one order by all of them."""
    M, N, K = 170, 136, 128
    a, b, w = rand(M, K, seed=1) + 1.0, rand(N, K, seed=2), rand(K, N, seed=3)
    for t in (b, w):
        A, B = (apart(a, step), t) if far == "A" else (a, apart(t, step))
        results = []
        if t is b:
            for ops in ((a, b), (A, B)):
                C = torch.empty(M, N, dtype=torch.bfloat16, device=DEV)
                strips = torch.full((hiplib.strip_stats_workspace(M, N),), float("nan"), device=DEV)
                hiplib.gemm(hiplib.NT, *ops, C, strip_stats=strips)
                results.append((C, strips))
        else:
            x, relu_out, skip = rand(M, N, seed=4), rand(M, N, seed=5), rand(M, N, seed=6)
            mean, rstd = torch.randn(2, N, generator=torch.Generator(device=DEV).manual_seed(7), device=DEV)
            for ops in ((a, w), (A, B)):
                C = torch.empty(M, N, dtype=torch.bfloat16, device=DEV)
                strips = torch.full((hiplib.bn_bwd_strips_workspace(M, N),), float("nan"), device=DEV)
                hiplib.gemm_bn_bwd(*ops, C, relu_out, x, mean, rstd, strips, resid=skip)
                results.append((C, strips))
        assert all(torch.equal(p, q) for p, q in zip(*results)) and not any(torch.isnan(p).any() for p in results[0])
