"""Products whose epilogue works on the accumulators in registers, and whose operands are reached by 32-bit offsets from a base
per tile: rows and columns off the tile, every epilogue kind, results in fp32, leading dimensions on either side of the limit."""
import pytest
import torch

pytestmark = pytest.mark.gpu
DEV = "cuda:0"


def rand(*shape, seed, scale=1.0):
    g = torch.Generator(device=DEV).manual_seed(seed)
    return (torch.randn(*shape, generator=g, device=DEV) * scale).bfloat16()


def framed(M, N, dtype=torch.bfloat16):
    wide = torch.full((M + 1, N + 8), 7.0, dtype=dtype, device=DEV)
    return wide, wide[:M, :N]


# tile the shape takes; a row or column group of a tile alone, whole tiles, some short of whole
@pytest.mark.parametrize("tile,M,N,K", [("64x64k64s4", 1, 8, 64), ("64x64k64s4", 33, 40, 128), ("64x64k64s4", 1050, 512, 192), ("k64s3", 2300, 1040, 448),
                                        ("128x128k64s3", 3301, 1032, 512), ("256x128k64s3", 8100, 1000, 512), ("256x128k64s3", 8192, 1024, 512)])
@pytest.mark.parametrize("layout", ["nt", "nn"])
def test_register_epilogue(hiplib, layout, tile, M, N, K):
    lay = hiplib.NT if layout == "nt" else hiplib.NN
    A, B = rand(M, K, seed=1), rand(*((N, K) if layout == "nt" else (K, N)), seed=2, scale=0.2)
    bias, X, R = rand(N, seed=3), rand(M, N, seed=4), rand(M, N, seed=5)
    wide, C = framed(M, N)
    wide2, D = framed(M, N)
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
    C1, D1 = (torch.full((M, N), 7.0, dtype=torch.bfloat16, device=DEV) for _ in range(2))
    hiplib.gemm(lay, A, B, C1, bias=bias, epilogue=hiplib.EPI_RESIDUAL, resid=R)
    near(C1, u + r)
    hiplib.gemm(lay, A, B, C1, epilogue=hiplib.EPI_MUL, aux_in=X)
    near(C1, prod * x, scale=x.abs())
    hiplib.gemm(lay, A, B, C1, epilogue=hiplib.EPI_MUL_POS, aux_in=X, resid=R)
    near(C1, torch.where(x > 0, prod + r, 0.0))
    hiplib.gemm(lay, A, B, C1, epilogue=hiplib.EPI_DACT, act=hiplib.ACT_RELU, aux_in=X)
    near(C1, torch.where(x > 0, prod, 0.0))
    hiplib.gemm(lay, A, B, C1, bias=bias, epilogue=hiplib.EPI_ACT, act=hiplib.ACT_RELU, aux_out=D1)
    near(D1, u)
    near(C1, u.clamp_min(0))
    hiplib.gemm(lay, A, B, C1, bias=bias, epilogue=hiplib.EPI_ACT_DACT, act=hiplib.ACT_GELU_TANH, aux_out=D1)
    g = u.clone().requires_grad_()
    y = torch.nn.functional.gelu(g, approximate="tanh")
    dy, = torch.autograd.grad(y.sum(), g)
    near(C1, y.detach(), scale=2.0)      # |gelu'| and |gelu''| stay below 1.2
    near(D1, dy.double(), scale=2.0)
    F0 = torch.randn(M, N, generator=torch.Generator(device=DEV).manual_seed(6), device=DEV)
    F = F0.clone()
    hiplib.gemm(lay, A, B, F, accumulate=True)
    assert ((F.double() - prod - F0.double()).abs() <= slack + 2.0 ** -23 * (prod.abs() + F0.double().abs() + 1.0)).all()


@pytest.mark.parametrize("layout", ["nt", "nn"])
def test_rows_far_apart(hiplib, layout):
    M, N, K, ld = 130, 136, 128, 1 << 22
    lay = hiplib.NT if layout == "nt" else hiplib.NN
    store = torch.empty(M * ld, dtype=torch.bfloat16, device=DEV)
    for step in (ld, ld - 8):
        A = store[: M * step].view(M, step)[:, :K]
        A.copy_(rand(M, K, seed=1))
        B = rand(*((N, K) if layout == "nt" else (K, N)), seed=2)
        C, D = (torch.empty(M, N, dtype=torch.bfloat16, device=DEV) for _ in range(2))
        variant = hiplib.gemm_variant(hiplib.gemm_desc(lay, A, B, C))
        assert variant.endswith("128x128k64r") == (step == ld)
        hiplib.gemm(lay, A, B, C)
        hiplib.gemm(lay, A.contiguous(), B, D)
        assert torch.equal(C, D)         # the kernels add up a contraction in one order
        hiplib.gemm_grouped([hiplib.gemm_desc(lay, A, B, C), hiplib.gemm_desc(lay, A, B, D)])
        assert torch.equal(C, D)
