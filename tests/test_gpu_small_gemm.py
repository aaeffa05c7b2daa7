"""bf16 GEMMs of few tiles (contraction dealt to the waves of a block) and weight gradients over row counts that are no
multiple of a k-tile, against fp64."""
import pytest
import torch

pytestmark = pytest.mark.gpu
DEV = "cuda:0"


def rand(*shape, seed, scale=1.0):
    g = torch.Generator().manual_seed(seed)
    return (torch.randn(*shape, generator=g) * scale).bfloat16().to(DEV)


def rel(got, ref):
    got, ref = got.double().cpu(), ref.double().cpu()
    return float((got - ref).abs().max() / ref.abs().max().clamp_min(1e-30))


# one slice, fewer slices than waves, ragged last slices, both slice widths, rows and columns off the tile, the largest
# single round (256 tiles) and a problem of more tiles that no DMA kernel takes
@pytest.mark.parametrize("M,N,K", [(64, 64, 8), (8, 8, 32), (72, 136, 40), (128, 384, 264), (65, 200, 1032), (65, 200, 64), (200, 8, 576), (1024, 1024, 96),
                                   (1000, 64, 1024), (20000, 64, 128), (3000, 64, 2056), (6000, 192, 72)])
@pytest.mark.parametrize("layout", ["nt", "nn"])
def test_products_of_few_tiles(hiplib, layout, M, N, K):
    lay = hiplib.NT if layout == "nt" else hiplib.NN
    A, B = rand(M, K, seed=1), rand(*((N, K) if layout == "nt" else (K, N)), seed=2, scale=0.2)
    bias, X = rand(N, seed=3), rand(M, N, seed=4)
    C, D = (torch.full((M, N), float("nan"), dtype=torch.bfloat16, device=DEV) for _ in range(2))
    variant = hiplib.gemm_variant(hiplib.gemm_desc(lay, A, B, C))
    assert variant.endswith("dma64x64k64s4" if K % 64 == 0 else "dma128x64s3" if (K, layout) == (96, "nt") else
                            "dma64x128s3" if K == 96 else "wave64x64k8" if M < 6000 else "wave64x64k4")
    prod = A.double().cpu() @ (B.double().cpu().t() if layout == "nt" else B.double().cpu())
    b, x = bias.double().cpu(), X.double().cpu()
    hiplib.gemm(lay, A, B, C, bias=bias, alpha=0.5)
    assert rel(C, 0.5 * prod + b) < 1e-2
    hiplib.gemm(lay, A, B, C, bias=bias, epilogue=hiplib.EPI_RESIDUAL, resid=X)
    assert rel(C, prod + b + x) < 1e-2
    hiplib.gemm(lay, A, B, C, epilogue=hiplib.EPI_MUL, aux_in=X)
    assert rel(C, prod * x) < 1e-2
    hiplib.gemm(lay, A, B, C, epilogue=hiplib.EPI_MUL_POS, aux_in=X, resid=D.fill_(0.25))
    assert rel(C, (prod + 0.25) * (x > 0)) < 1e-2
    hiplib.gemm(lay, A, B, C, bias=bias, epilogue=hiplib.EPI_ACT_DACT, act=hiplib.ACT_RELU, aux_out=D)
    u = prod + b
    assert rel(C, u.clamp_min(0)) < 1e-2
    assert float((D.double().cpu() != (u > 0)).double().mean()) < 2e-3     # pre-activations that round to the other side of zero
    G0 = torch.randn(M, N, generator=torch.Generator().manual_seed(5)).to(DEV)
    G = G0.clone()
    hiplib.gemm(lay, A, B, G, accumulate=True)
    assert rel(G, G0.double().cpu() + prod) < 1e-4
    G2 = G0.clone()
    hiplib.gemm(lay, A, B, G2, accumulate=True)
    assert torch.equal(G, G2)


# (rows, shapes of dy and x): few tiles (eight waves a tile), up to four tiles a CU (four waves), 128x128 tiles
@pytest.mark.parametrize("rows,shapes", [(1, [(64, 64), (8, 72)]), (31, [(128, 128), (384, 128)]), (1050, [(192, 768), (576, 192)]),
                                         (333, [(512, 2048), (2048, 512), (512, 512)]), (2049, [(1024, 4096), (4096, 1024)]),
                                         (95, [(1024, 4096), (4096, 1024)])])
def test_weight_gradients_over_ragged_rows(hiplib, rows, shapes):
    descs, want = [], []
    for i, (m, n) in enumerate(shapes):
        dy, x = rand(rows, m, seed=10 + i), rand(rows, n, seed=20 + i)
        g, b = torch.full((m, n), 0.5, device=DEV), torch.full((m,), -1.0, device=DEV)
        ws = torch.empty(hiplib.colsum_workspace(max(m, n)), device=DEV)
        descs.append((hiplib.gemm_desc(hiplib.TN, dy, x, g, accumulate=True, colsum_out=b, colsum_ws=ws), dy, x, g, b))
        want.append((dy.double().cpu().t() @ x.double().cpu() + 0.5, dy.double().cpu().sum(0) - 1.0))
    hiplib.gemm_grouped([d[0] for d in descs])
    for (_, dy, x, g, b), (wg, wb) in zip(descs, want):
        assert rel(g, wg) < 1e-5 and rel(b, wb) < 1e-5
    # one by one: the kernel may be another, the sums are the same up to their order
    for (_, dy, x, g, b), (wg, wb) in zip(descs, want):
        g1, b1 = torch.full_like(g, 0.5), torch.full_like(b, -1.0)
        hiplib.gemm(hiplib.TN, dy, x, g1, accumulate=True, colsum_out=b1, colsum_ws=torch.empty(hiplib.colsum_workspace(max(g.shape)), device=DEV))
        assert rel(g1, wg) < 1e-5 and rel(b1, wb) < 1e-5


@pytest.mark.parametrize("n,h,w,c,co", [(3, 9, 7, 128, 128), (1, 11, 13, 64, 64), (5, 31, 15, 192, 64), (7, 6, 40, 64, 512),
                                        (1, 9, 9, 512, 512), (9, 23, 23, 256, 640)])
def test_conv_weight_gradient_over_ragged_pixels(hiplib, n, h, w, c, co):
    """The patch-matrix operand gathered inside the kernel, pixels no multiple of the k-tile, whole and split."""
    R = n * h * w
    dy, x = rand(R, co, seed=1), rand(R, c, seed=2)
    col = torch.empty(R, 9 * c, dtype=torch.bfloat16, device=DEV)
    hiplib.patch3x3(x, col, n, h, w, c)
    want = dy.double().cpu().t() @ col.double().cpu()
    for ws in (None, torch.empty(8 * co * 9 * c, device=DEV)):
        g = torch.zeros(co, 9 * c, device=DEV)
        hiplib.gemm_grouped([hiplib.gemm_desc(hiplib.TN, dy, x, g, accumulate=True, conv=(h, w))], splitk_ws=ws)
        assert rel(g, want) < 1e-5
