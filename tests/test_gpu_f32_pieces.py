"""fp32 products on bf16 matrix instructions: both tiles, every layout, rows, columns and contractions off the tile, against fp64 -- no further
from it than the fp32 instructions are --, every epilogue, and operands that are not finite or too large for bf16."""
import pytest
import torch

pytestmark = pytest.mark.gpu
DEV = "cuda:0"


def rand(*shape, seed, scale=1.0):
    g = torch.Generator(device=DEV).manual_seed(seed)
    return torch.randn(*shape, generator=g, device=DEV) * scale


def operands(layout, M, N, K):
    a, b = rand(*((K, M) if layout == "tn" else (M, K)), seed=1), rand(*((N, K) if layout == "nt" else (K, N)), seed=2)
    return a, b, (a.double().t() if layout == "tn" else a.double()).contiguous(), (b.double().t() if layout == "nt" else b.double()).contiguous()


def off(c, ref):
    return float((c.double() - ref).norm() / ref.norm())


CASES = [("nt", 4100, 2060, 260, 128), ("nt", 2044, 776, 772, 64), ("nn", 4100, 2060, 264, 128), ("nn", 2044, 776, 780, 64), ("tn", 2044, 1036, 1051, 128),
         ("tn", 2048, 2048, 256, 128)]


@pytest.mark.parametrize("layout,M,N,K,tile", CASES)
def test_products(hiplib, layout, M, N, K, tile):
    lay = getattr(hiplib, layout.upper())
    a, b, a64, b64 = operands(layout, M, N, K)
    wide = torch.full((M + 1, N + 8), 7.0, device=DEV)
    C, F = wide[:M, :N], torch.empty(M, N, device=DEV)
    assert hiplib.gemm_variant(hiplib.gemm_desc(lay, a, b, C, pieces=True)) == f"f32_{layout}_pieces128x{tile}"
    assert "pieces" not in hiplib.gemm_variant(hiplib.gemm_desc(lay, a, b, C))
    hiplib.gemm(lay, a, b, C, pieces=True)
    hiplib.gemm(lay, a, b, F)
    ref = a64 @ b64
    assert (wide[M:] == 7).all() and (wide[:, N:] == 7).all()
    assert off(C, ref) <= off(F, ref)
    # six products a k, each rounded once at most, and the three left out, below 2^-24 of the product each
    size = a64.abs() @ b64.abs()
    assert ((C.double() - ref).abs() <= (K + 3) * 2.0 ** -24 * size).all()
    C2 = torch.empty(M, N, device=DEV)
    hiplib.gemm(lay, a, b, C2, pieces=True)
    assert torch.equal(C, C2)
    F = torch.ones(M, N, device=DEV)
    hiplib.gemm(lay, a, b, F, pieces=True, accumulate=True, alpha=0.5)
    assert ((F.double() - 1.0 - 0.5 * ref).abs() <= K * 2.0 ** -24 * size + 2.0 ** -23 * (ref.abs() + 2.0)).all()


@pytest.mark.parametrize("layout,M,N,K,tile", CASES[:5])
@pytest.mark.parametrize("of_a,of_b", [((-126, -112), (40, 60)), ((50, 60), (-126, -120)), ((-149, -126), (60, 80)), ((-70, -55), (-70, -60)), ((-126, 60), (-20, 20)),
                                       ((44, 49), (44, 49)), ((100, 115), (-30, 0))])
def test_powers_of_two(hiplib, layout, M, N, K, tile, of_a, of_b):
    """Values of every size fp32 has, the smallest ones and subnormals (against large ones) among them: within the bound of test_products, no further from fp64
    than the fp32 instructions, also where the scaled sums leave fp32's range and are made again."""
    lay = getattr(hiplib, layout.upper())
    a, b, _, _ = operands(layout, M, N, K)
    for x, (lo, hi), seed in ((a, of_a, 11), (b, of_b, 12)):
        g = torch.Generator(device=DEV).manual_seed(seed)
        x.copy_(x.double() * 2.0 ** torch.randint(lo, hi + 1, x.shape, generator=g, device=DEV).double())
    a64, b64 = (a.double().t() if layout == "tn" else a.double()).contiguous(), (b.double().t() if layout == "nt" else b.double()).contiguous()
    C, F = torch.empty(M, N, device=DEV), torch.empty(M, N, device=DEV)
    hiplib.gemm(lay, a, b, C, pieces=True)
    hiplib.gemm(lay, a, b, F)
    ref, size = a64 @ b64, a64.abs() @ b64.abs()
    # (a product or sum below 2^-126 is rounded to a multiple of 2^-149 by either)
    assert ((C.double() - ref).abs() <= (K + 3) * (2.0 ** -24 * size + 2.0 ** -150)).all()
    # Values of up to 20 octaves in either operand: no further from fp64 than the fp32 instructions.  1 %: where all is made again it is the same arithmetic in
    # another order.  (Of many more, one product is most of a sum, which fp32 then rounds once, and the bf16 instruction drops what lies below the
    # last bit of the largest of its addends: up to a quarter further off than fp32, within the bound above.)
    if max(of_a[1] - of_a[0], of_b[1] - of_b[0]) <= 23:
        assert off(C, ref) <= 1.01 * off(F, ref)


@pytest.mark.parametrize("layout,M,N,K,tile", CASES[:4])
def test_epilogues(hiplib, layout, M, N, K, tile):
    """Against the same epilogue on the fp32 instructions: both products lie within the bound of test_products of the exact one, and what is
    made of them moves by at most 2.3 times as much (GELU and its derivative, a factor of the residual kinds below 4 standard deviations)."""
    lay = getattr(hiplib, layout.upper())
    a, b, a64, b64 = operands(layout, M, N, K)
    slack = 2 * 2.3 * K * 2.0 ** -24 * (a64.abs() @ b64.abs()) + 1e-6
    bias, x, r = rand(N, seed=3), rand(M, N, seed=4).clamp(-2.3, 2.3), rand(M, N, seed=5)
    kinds = [dict(bias=bias), dict(bias=bias, epilogue=hiplib.EPI_RESIDUAL, resid=r), dict(epilogue=hiplib.EPI_MUL, aux_in=x),
             dict(epilogue=hiplib.EPI_MUL_POS, aux_in=x), dict(epilogue=hiplib.EPI_MUL_POS, aux_in=x, resid=r), dict(epilogue=hiplib.EPI_DACT, act=hiplib.ACT_GELU_TANH, aux_in=x),
             dict(bias=bias, epilogue=hiplib.EPI_ACT, act=hiplib.ACT_GELU_TANH), dict(bias=bias, epilogue=hiplib.EPI_ACT_DACT, act=hiplib.ACT_GELU_TANH, aux_out=None)]
    if layout == "nt":
        kinds += [dict(bias=bias, dropout=(0.1, (7, 9)), epilogue=hiplib.EPI_RESIDUAL, resid=r), dict(bias=bias, dropout=(0.1, (7, 9)))]
    for kw in kinds:
        out = []
        for pieces in (True, False):
            c, d = torch.full((M, N), 7.0, device=DEV), torch.full((M, N), 7.0, device=DEV)
            hiplib.gemm(lay, a, b, c, pieces=pieces, **{k: d if k == "aux_out" else v for k, v in kw.items()})
            out.append((c.double(), d.double()))
        (c, d), (c0, d0) = out
        assert ((c - c0).abs() <= slack).all() and ((d - d0).abs() <= slack).all(), kw


@pytest.mark.parametrize("layout,M,N,K,tile", CASES[:5])
def test_values_that_bf16_does_not_hold(hiplib, layout, M, N, K, tile):
    """Infinities, NaN and values that round to more than the largest bf16: what fp32 arithmetic makes of them, in their row or column only."""
    lay = getattr(hiplib, layout.upper())
    a, b, _, _ = operands(layout, M, N, K)
    av, bv = (a.t() if layout == "tn" else a), (b.t() if layout == "nt" else b)
    av[3, 5], av[130, K - 1], av[M - 1, 0], bv[7, N - 2] = float("inf"), float("nan"), 3.4e38, -float("inf")
    bv[0] *= 1e-3
    C = torch.empty(M, N, device=DEV)
    hiplib.gemm(lay, a, b, C, pieces=True)
    ref = av.double().contiguous() @ bv.double().contiguous()
    assert torch.equal(torch.isnan(C), torch.isnan(ref)) and torch.equal(torch.isinf(C), torch.isinf(ref))
    ok = torch.isfinite(ref)
    size = torch.nan_to_num(av.double().abs(), 0, 0).contiguous() @ torch.nan_to_num(bv.double().abs(), 0, 0).contiguous()
    assert ((C.double() - ref).abs()[ok] <= (K * 2.0 ** -24 * size)[ok]).all() and (C.double() == ref)[torch.isinf(ref)].all()


def test_grouped_weight_gradients(hiplib):
    """A layer's, with their bias gradients: against fp64, and nearer to it than without pieces."""
    R, h = 1043, 512
    dy = [rand(R, n, seed=10 + i) for i, n in enumerate((3 * h, h, 4 * h, h))]
    x = [rand(R, n, seed=20 + i) for i, n in enumerate((h, h, h, 4 * h))]
    outs = []
    for pieces in (True, False):
        g, s = [torch.ones(d.shape[1], v.shape[1], device=DEV) for d, v in zip(dy, x)], [torch.ones(d.shape[1], device=DEV) for d in dy]
        ws = [torch.empty(hiplib.colsum_workspace(d.shape[1]), device=DEV) for d in dy]
        descs = [hiplib.gemm_desc(hiplib.TN, d, v, G, accumulate=True, colsum_out=c, colsum_ws=w, pieces=pieces) for d, v, G, c, w in zip(dy, x, g, s, ws)]
        hiplib.gemm_grouped(descs)
        outs.append((g, s))
    for i, (d, v) in enumerate(zip(dy, x)):
        ref = 1.0 + d.double().t().contiguous() @ v.double()
        size = d.double().abs().t().contiguous() @ v.double().abs() + 1.0
        assert ((outs[0][0][i].double() - ref).abs() <= (R + 3) * 2.0 ** -24 * size).all()
        assert off(outs[0][0][i], ref) < off(outs[1][0][i], ref)       # (the pieces were taken)
        assert torch.equal(outs[0][1][i], outs[1][1][i])


@pytest.mark.parametrize("layout,M,N,K", [("nt", 2048, 3072, 768), ("nn", 2048, 768, 3072), ("tn", 3072, 768, 2048)])
def test_time_of_values_that_bf16_does_not_hold(hiplib, layout, M, N, K):
    """A product that is made again costs the fp32 instructions' time beside its own, not a multiple: all of it (a diverged step), or what one row
    spoils.  (Measured: at most 3 times; 6 leaves room for a slow clock.)"""
    lay = getattr(hiplib, layout.upper())
    a, b, _, _ = operands(layout, M, N, K)
    C = torch.empty(M, N, device=DEV)
    one, every = a.clone(), torch.full_like(a, float("nan"))
    one[3, 5] = float("nan")

    def least(x):
        times = []
        for _ in range(8):
            start, end = torch.cuda.Event(enable_timing=True), torch.cuda.Event(enable_timing=True)
            start.record()
            for _ in range(4):
                hiplib.gemm(lay, x, b, C, pieces=True)
            end.record()
            torch.cuda.synchronize()
            times.append(start.elapsed_time(end))
        return min(times)

    finite = least(a)
    assert least(one) <= 6 * finite and least(every) <= 6 * finite


def test_problems_that_fp32_instructions_do_sooner(hiplib):
    """What the rounds of the tiles leave to the fp32 kernels, bit for bit: a product of one half-filled round, the weight gradients of a layer 576 wide over
    1077 rows (275 tiles on 256 CUs: 109 us on pieces, 88) and of one 832 wide over 256 (70, 57)."""
    a, b, _, _ = operands("nn", 1305, 1536, 384)
    C, F = torch.empty(1305, 1536, device=DEV), torch.empty(1305, 1536, device=DEV)
    hiplib.gemm(hiplib.NN, a, b, C, pieces=True)
    hiplib.gemm(hiplib.NN, a, b, F)
    assert torch.equal(C, F)
    for h, R in ((576, 1077), (832, 256)):
        ops = [(rand(R, m, seed=m), rand(R, n, seed=n + 1)) for m, n in ((3 * h, h), (h, h), (4 * h, h), (h, 4 * h))]
        outs = []
        for pieces in (True, False):
            g = [torch.zeros(d.shape[1], v.shape[1], device=DEV) for d, v in ops]
            hiplib.gemm_grouped([hiplib.gemm_desc(hiplib.TN, d, v, G, accumulate=True, pieces=pieces) for (d, v), G in zip(ops, g)])
            outs.append(g)
        assert all(torch.equal(p, q) for p, q in zip(*outs))
