"""GEMMs of few tiles (contraction dealt to the waves of a block) and weight gradients over row counts that are no
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


# More 64x64 tiles than two a CU and a contraction that ends inside a k-tile: k-tiles of 8 to 56, one k-tile in all, rows and
# columns off the tile.  bf16 results: half an ulp, at most 2^-8 of |C|, beside the fp32 sums' K eps sum |a b|.
@pytest.mark.parametrize("M,N,K", [(3001, 1000, 8), (4100, 520, 40), (2100, 1096, 72), (33000, 72, 88), (2049, 1032, 1000), (96, 33000, 136)])
@pytest.mark.parametrize("layout", ["nt", "nn"])
def test_large_products_of_ragged_contractions(hiplib, layout, M, N, K):
    lay = hiplib.NT if layout == "nt" else hiplib.NN
    A, B = rand(M, K, seed=1), rand(*((N, K) if layout == "nt" else (K, N)), seed=2)
    wide = torch.full((M + 1, N + 8), 7.0, dtype=torch.bfloat16, device=DEV)
    C = wide[:M, :N]
    assert hiplib.gemm_variant(hiplib.gemm_desc(lay, A, B, C)).endswith("dma128x128k64r")
    hiplib.gemm(lay, A, B, C)
    a, b = A.double(), (B.double().t() if layout == "nt" else B.double()).contiguous()
    want, slack = a @ b, K * 2.0 ** -24 * (a.abs() @ b.abs())
    assert ((C.double() - want).abs() <= 2.0 ** -8 * (want.abs() + slack) + slack).all()
    assert (wide[M:] == 7).all() and (wide[:, N:] == 7).all()       # nothing written past the rows and columns
    bias, X = rand(N, seed=3), rand(M, N, seed=4)
    R = torch.empty(M, N, dtype=torch.bfloat16, device=DEV)
    hiplib.gemm(lay, A, B, R, bias=bias, epilogue=hiplib.EPI_RESIDUAL, resid=X, alpha=0.5)
    assert rel(R, 0.5 * want + bias.double() + X.double()) < 1e-2
    if layout == "nt":      # as a member of a group it runs by itself; with dropout, the kernel that decides
        C2, C3 = torch.empty(M, N, dtype=torch.bfloat16, device=DEV), torch.empty(M, N, dtype=torch.bfloat16, device=DEV)
        hiplib.gemm_grouped([hiplib.gemm_desc(lay, A, B, C2), hiplib.gemm_desc(lay, A, B, C3)])
        assert torch.equal(C, C2) and torch.equal(C, C3)
        key = hiplib.dropout_key(1, 2, 3, 4, 5)
        hiplib.gemm(lay, A, B, C2, dropout=(0.25, key))
        hiplib.dropout_apply(C3, C3, 0.25, key)
        assert torch.equal(C2 == 0, C3 == 0) and rel(C2, C3) < 1e-2     # two roundings against one


# heads of a width that the fused attention does not take: the products of a materialised attention, forward and backward
@pytest.mark.parametrize("b,h,s,d", [(3, 12, 520, 72), (1, 24, 1032, 40), (2, 20, 456, 80)])
def test_attention_products_of_ragged_lengths(hiplib, b, h, s, d):
    P, X = rand(b, h, s, s, seed=1), rand(b * s, 3 * h * d, seed=2)
    heads = X.view(b, s, 3, h, d).permute(2, 0, 3, 1, 4).double()      # [3, b, h, s, d]
    sp, sx = (h * s * s, s * s), (s * 3 * h * d, d)
    at = lambda t, i: t.data_ptr() + i * h * d * t.element_size()
    for lay, want in ((hiplib.NN, P.double() @ heads[1].contiguous()), (hiplib.TN, P.double().transpose(2, 3).contiguous() @ heads[1].contiguous())):
        out = torch.full_like(X, 7.0)
        hiplib.gemm_batched(lay, hiplib.BF16, s, d, s, P.data_ptr(), s, sp, at(X, 1), 3 * h * d, sx, at(out, 2), 3 * h * d, sx, b, h)
        got = out.view(b, s, 3, h, d).permute(2, 0, 3, 1, 4)
        assert rel(got[2], want) < 1e-2 and (got[:2] == 7).all()
    S = torch.empty(b, h, s, s, dtype=torch.bfloat16, device=DEV)
    hiplib.gemm_batched(hiplib.NT, hiplib.BF16, s, s, d, at(X, 0), 3 * h * d, sx, at(X, 1), 3 * h * d, sx, S.data_ptr(), s, sp, b, h)
    assert rel(S, heads[0].contiguous() @ heads[1].transpose(2, 3).contiguous()) < 1e-2


# (rows, shapes of dy and x): few tiles (eight waves a tile), up to four tiles a CU (four waves), 128x128 tiles
@pytest.mark.parametrize("rows,shapes", [(1, [(64, 64), (8, 72)]), (31, [(128, 128), (384, 128)]), (1050, [(192, 768), (576, 192)]),
                                         (333, [(512, 2048), (2048, 512), (512, 512)]), (2049, [(1024, 4096), (4096, 1024)]),
                                         (95, [(1024, 4096), (4096, 1024)]), (100, [(33000, 72), (72, 33000)])])
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


# One slice and a part of one, a ragged last slice, all four slices whole; fewer rows or columns than a tile, remainders, the
# largest the rule takes (1024 tiles).  Sums of K products in fp32, K roundings at most: |error| <= K eps sum |a b| (eps = 2^-24).
@pytest.mark.parametrize("M,N,K", [(4, 4, 4), (36, 28, 32), (32, 32, 36), (100, 72, 100), (128, 384, 128), (64, 128, 64), (8, 1024, 124),
                                   (1024, 1024, 96)])
@pytest.mark.parametrize("layout", ["nt", "nn", "tn"])
def test_fp32_products_of_few_tiles(hiplib, layout, M, N, K):
    lay = {"nt": hiplib.NT, "nn": hiplib.NN, "tn": hiplib.TN}[layout]
    mk = lambda *shape, seed: torch.randn(*shape, generator=torch.Generator().manual_seed(seed)).to(DEV)
    A, B = mk(*((K, M) if layout == "tn" else (M, K)), seed=1), mk(*((N, K) if layout == "nt" else (K, N)), seed=2)
    bias, X, G = mk(N, seed=3), mk(M, N, seed=4), mk(M, N, seed=5)
    a, b = A.double().cpu(), B.double().cpu()
    a, b = a.t() if layout == "tn" else a, b.t() if layout == "nt" else b
    prod, bound = a @ b, (K + 4) * 2.0 ** -24 * (a.abs() @ b.abs() + bias.double().cpu().abs() + X.double().cpu().abs() + G.double().cpu().abs())
    C = torch.full((M, N), float("nan"), device=DEV)
    few = layout == "nn" or layout == "tn" and M * N < 1024 * 1024     # (a forward product keeps the larger tiles' order)
    assert hiplib.gemm_variant(hiplib.gemm_desc(lay, A, B, C)).endswith("wave32x32k4" if few else "64x64")
    hiplib.gemm(lay, A, B, C, bias=bias, epilogue=hiplib.EPI_RESIDUAL, resid=X)
    assert bool(((C.double().cpu() - (prod + bias.double().cpu() + X.double().cpu())).abs() <= bound).all())
    acc = G.clone()
    hiplib.gemm(lay, A, B, acc, accumulate=True)
    assert bool(((acc.double().cpu() - (prod + G.double().cpu())).abs() <= bound).all())
    if layout == "nt":
        hiplib.gemm(lay, A, B, C, bias=bias, epilogue=hiplib.EPI_ACT_DACT, act=hiplib.ACT_RELU, aux_out=X)
        u = prod + bias.double().cpu()
        assert bool(((C.double().cpu() - u.clamp_min(0)).abs() <= bound).all()) and bool(((X.double().cpu() == (u > 0)) | (u.abs() <= bound)).all())
    # a layer's problems in one launch give the bits they give alone, also beside one of many tiles
    if layout == "tn":
        for other in (64, 1024):
            A2, one, two = mk(K, other, seed=6), G.clone(), torch.zeros(other, N, device=DEV)
            big = torch.zeros(other, N, device=DEV)
            hiplib.gemm(lay, A2, B, big, accumulate=True)
            hiplib.gemm_grouped([hiplib.gemm_desc(lay, A, B, one, accumulate=True), hiplib.gemm_desc(lay, A2, B, two, accumulate=True)])
            assert bool(((one.double().cpu() - (prod + G.double().cpu())).abs() <= bound).all())
            if other == 64 and M * N < 1024 * 1024:
                assert torch.equal(one, acc) and torch.equal(two, big)


# the products of attention heads inside a [rows, 3 h] buffer, as one batched launch of few tiles
@pytest.mark.parametrize("b,heads,seq", [(1, 1, 36), (2, 3, 64), (4, 2, 100), (1, 2, 512)])
def test_fp32_batched_heads_of_few_tiles(hiplib, b, heads, seq):
    d = 64
    h = heads * d
    qkv = torch.randn(b * seq, 3 * h, generator=torch.Generator().manual_seed(9)).to(DEV)
    P = torch.empty(b, heads, seq, seq, device=DEV)
    hiplib.gemm_batched(hiplib.NT, hiplib.dtype_code(torch.float32), seq, seq, d, qkv.data_ptr(), 3 * h, (seq * 3 * h, d), qkv.data_ptr() + 4 * h,
                        3 * h, (seq * 3 * h, d), P.data_ptr(), seq, (heads * seq * seq, seq * seq), b, heads, alpha=0.125)
    q, k = (qkv[:, i * h:(i + 1) * h].double().cpu().view(b, seq, heads, d).transpose(1, 2) for i in (0, 1))
    bound = (d + 2) * 2.0 ** -24 * 0.125 * (q.abs() @ k.abs().transpose(-1, -2))
    assert bool(((P.double().cpu() - 0.125 * q @ k.transpose(-1, -2)).abs() <= bound).all())


# the first row pitch that the 32-bit offsets inside a tile are not used for, and one where 64 rows pass 2^32 bytes; K with and
# without a ragged last k-tile.  |error| <= K eps sum |a b|, as above.
@pytest.mark.parametrize("ld", [1 << 22, (1 << 24) + (1 << 20) + 4])
@pytest.mark.parametrize("layout,M,N,K", [("nt", 70, 36, 64), ("nt", 3, 64, 100), ("nn", 66, 68, 44), ("tn", 64, 72, 40)])
def test_fp32_rows_of_any_pitch(hiplib, layout, M, N, K, ld):
    lay = {"nt": hiplib.NT, "nn": hiplib.NN, "tn": hiplib.TN}[layout]
    g = torch.Generator().manual_seed(3)
    shapes = ((K, M) if layout == "tn" else (M, K), (N, K) if layout == "nt" else (K, N))
    host = [torch.randn(s, generator=g) for s in shapes]
    A, B = [torch.as_strided(torch.empty((t.shape[0] - 1) * ld + t.shape[1], device=DEV), t.shape, (ld, 1)).copy_(t) for t in host]
    C, C2, C3 = (torch.full((M, N), float("nan"), device=DEV) for _ in range(3))
    descs = [hiplib.gemm_desc(lay, A, B, c) for c in (C, C2, C3)]
    assert hiplib.gemm_variant(descs[0]).endswith("64x64wide")
    hiplib.gemm(lay, A, B, C)
    hiplib.gemm_grouped(descs[1:])
    a, b = host[0].double(), host[1].double()
    a, b = (a.t() if layout == "tn" else a), (b.t() if layout == "nt" else b)
    bound = K * 2.0 ** -24 * (a.abs() @ b.abs())
    assert ((C.double().cpu() - a @ b).abs() <= bound).all() and torch.equal(C, C2) and torch.equal(C, C3)


# Products of few tiles against the same rows inside a product of many, which the larger tiles run: the same bits.  Contractions of
# a part of a k-tile, around 64, around the four stages of the ring, and long ones that two groups share; rows and columns of
# less than a tile, with remainders, and the most tiles the rule takes (128).  (NN with at most 128 columns of contraction is the
# 32x32 wave tiles': test_fp32_products_of_few_tiles.  Its shortest here fill three of the ring's four stages.)
QUARTER = [(4, 4, 4), (32, 36, 60), (33, 64, 64), (70, 100, 68), (128, 128, 252), (100, 72, 256), (64, 260, 260), (512, 900, 320),
           (36, 28, 512), (70, 132, 524), (130, 64, 580), (1024, 512, 1036)]


@pytest.mark.parametrize("layout,M,N,K", [("nt", *s) for s in QUARTER] + [("nn", *s) for s in QUARTER if s[2] > 128] +
                         [("nn", 4, 4, 132), ("nn", 33, 64, 188), ("nn", 70, 100, 192), ("nn", 32, 36, 196)])
def test_fp32_quarter_tiles_have_the_bits_of_whole_ones(hiplib, layout, M, N, K):
    lay = hiplib.NT if layout == "nt" else hiplib.NN
    mk = lambda *shape, seed: torch.randn(*shape, generator=torch.Generator().manual_seed(seed)).to(DEV)
    rows = max(M, 64 * (130 * 64 // N + 1))     # more than 128 tiles, fewer than the 512 from which on no contraction is shared
    A, B = mk(rows, K, seed=1), mk(*((N, K) if layout == "nt" else (K, N)), seed=2)
    bias, X, G = mk(N, seed=3), mk(rows, N, seed=4), mk(rows, N, seed=5)
    few, many = hiplib.gemm_variant(hiplib.gemm_desc(lay, A[:M], B, G[:M])), hiplib.gemm_variant(hiplib.gemm_desc(lay, A, B, G))
    assert few == many.replace("64x", "quarter64x", 1) and "quarter" not in many
    for kw in (dict(bias=bias, epilogue=hiplib.EPI_RESIDUAL), dict(epilogue=hiplib.EPI_ACT_DACT, act=hiplib.ACT_GELU_TANH), dict(accumulate=True, alpha=0.5),
               dict(epilogue=hiplib.EPI_MUL_POS)):
        out = []
        for m in (M, rows):
            C, aux = G[:m].clone(), X[:m].clone()
            extra = {hiplib.EPI_RESIDUAL: dict(resid=aux), hiplib.EPI_ACT_DACT: dict(aux_out=aux), hiplib.EPI_MUL_POS: dict(aux_in=aux, resid=G[:m])}
            hiplib.gemm(lay, A[:m], B, C, **kw, **extra.get(kw.get("epilogue"), {}))
            out.append((C[:M], aux[:M]))
        assert torch.equal(out[0][0], out[1][0]) and torch.equal(out[0][1], out[1][1]), kw
    prod = A[:M].double().cpu() @ (B.double().cpu().t() if layout == "nt" else B.double().cpu())
    C = torch.full((M, N), float("nan"), device=DEV)
    hiplib.gemm(lay, A[:M], B, C)
    bound = K * 2.0 ** -24 * (A[:M].double().cpu().abs() @ (B.double().cpu().t() if layout == "nt" else B.double().cpu()).abs())
    assert bool(((C.double().cpu() - prod).abs() <= bound).all())


# 128x128 tiles of three stages, whose loop reads fragments a k-tile ahead, against the same rows inside a product of tiles that do
# not: the same bits, for odd and even numbers of k-tiles; ragged rows and columns.
@pytest.mark.parametrize("layout", ["nt", "nn"])
@pytest.mark.parametrize("K", [512, 576, 640, 704, 832])
def test_128_tiles_that_read_ahead_have_the_bits_of_others(hiplib, K, layout):
    lay, M, N, rows = getattr(hiplib, layout.upper()), 5500, 616, 14000
    A, B = rand(rows, K, seed=1), rand(*((N, K) if layout == "nt" else (K, N)), seed=2, scale=0.2)
    bias, X, R = rand(N, seed=3), rand(rows, N, seed=4), rand(rows, N, seed=5)
    names = [hiplib.gemm_variant(hiplib.gemm_desc(lay, A[:m], B, X[:m])) for m in (M, rows)]
    assert names[0].endswith("dma128x128k64s3") and names[1].endswith(("dma256x256k64", "dma256x192k64", "dma256x256w8db")), names
    for kw in (dict(bias=bias), dict(bias=bias, epilogue=hiplib.EPI_RESIDUAL), dict(epilogue=hiplib.EPI_MUL), dict(epilogue=hiplib.EPI_MUL_POS),
               dict(bias=bias, epilogue=hiplib.EPI_ACT_DACT, act=hiplib.ACT_GELU_TANH), dict(bias=bias, dropout=(0.1, (7, 9)))):
        if "dropout" in kw and layout == "nn":
            continue
        out = []
        for m in (M, rows):
            C, aux = torch.full((m, N), float("nan"), dtype=torch.bfloat16, device=DEV), X[:m].clone()
            extra = {hiplib.EPI_RESIDUAL: dict(resid=aux), hiplib.EPI_MUL: dict(aux_in=aux), hiplib.EPI_MUL_POS: dict(aux_in=aux, resid=R[:m]),
                     hiplib.EPI_ACT_DACT: dict(aux_out=aux)}
            hiplib.gemm(lay, A[:m], B, C, **kw, **extra.get(kw.get("epilogue"), {}))
            out.append((C[:M], aux[:M]))
        assert torch.equal(out[0][0], out[1][0]) and torch.equal(out[0][1], out[1][1]), kw
    prod = A[:M].float() @ (B.float().t() if layout == "nt" else B.float())
    C = torch.empty(M, N, dtype=torch.bfloat16, device=DEV)
    hiplib.gemm(lay, A[:M], B, C)
    assert rel(C, prod) < 2.0 ** -8      # half an ulp of bf16, and the sums' K eps


# The small tiles' loop against the same rows inside a product that 256x128 tiles run: the same bits.  One k-tile, as many as the
# ring has stages and one more, odd and even numbers of them beyond; rows off the tile; every epilogue that fetches an operand.
@pytest.mark.parametrize("K", [64, 128, 192, 256, 320, 448, 576])
@pytest.mark.parametrize("M,tile", [(100, "64x64k64s4"), (2050, "128x64k64s3"), (2050, "64x128k64s3")])
def test_small_tiles_have_the_bits_of_large_ones(hiplib, M, tile, K):
    lay, N, rows = (hiplib.NN, 640, 8200) if tile == "64x128k64s3" else (hiplib.NT, 640, 8200)
    A, B = rand(rows, K, seed=1), rand(*((N, K) if lay == hiplib.NT else (K, N)), seed=2, scale=0.2)
    bias, X, R = rand(N, seed=3), rand(rows, N, seed=4), rand(rows, N, seed=5)
    names = [hiplib.gemm_variant(hiplib.gemm_desc(lay, A[:m], B, X[:m])) for m in (M, rows)]
    if K > 64:
        assert names[0].endswith(tile) and names[1].endswith("dma256x128k64s3" if K >= 256 or lay == hiplib.NN else "dma128x64k64s3"), names
    for kw in (dict(bias=bias), dict(bias=bias, epilogue=hiplib.EPI_RESIDUAL), dict(epilogue=hiplib.EPI_MUL), dict(epilogue=hiplib.EPI_MUL_POS),
               dict(bias=bias, epilogue=hiplib.EPI_ACT_DACT, act=hiplib.ACT_GELU_TANH), dict(bias=bias, dropout=(0.1, (7, 9)))):
        if "dropout" in kw and lay != hiplib.NT:
            continue
        out = []
        for m in (M, rows):
            C, aux = torch.full((m, N), float("nan"), dtype=torch.bfloat16, device=DEV), X[:m].clone()
            extra = {hiplib.EPI_RESIDUAL: dict(resid=aux), hiplib.EPI_MUL: dict(aux_in=aux), hiplib.EPI_MUL_POS: dict(aux_in=aux, resid=R[:m]),
                     hiplib.EPI_ACT_DACT: dict(aux_out=aux)}
            hiplib.gemm(lay, A[:m], B, C, **kw, **extra.get(kw.get("epilogue"), {}))
            out.append((C[:M], aux[:M]))
        assert torch.equal(out[0][0], out[1][0]) and torch.equal(out[0][1], out[1][1]), kw
    prod = A[:M].double().cpu() @ (B.double().cpu().t() if lay == hiplib.NT else B.double().cpu())
    C = torch.empty(M, N, dtype=torch.bfloat16, device=DEV)
    hiplib.gemm(lay, A[:M], B, C)
    assert rel(C, prod) < 2.0 ** -8      # half an ulp of bf16, and the sums' K eps


# Weight gradients whose 128x128 tiles fill a round, three a CU: in lock step from 8192 rows on, free below, ragged and whole
# contractions; against each problem by itself (the same k order, free): the same bits, bias gradients too.
@pytest.mark.parametrize("rows", [8184, 8192, 8201])
def test_weight_gradients_of_a_full_round(hiplib, rows):
    shapes = [(3072, 1024), (2048, 1024), (3584, 1024), (1024, 3584)]
    ops = [(rand(rows, m, seed=2 * i), rand(rows, n, seed=2 * i + 1)) for i, (m, n) in enumerate(shapes)]
    runs = []
    for grouped in (True, False):
        C, bias = [torch.ones(m, n, device=DEV) for m, n in shapes], [torch.ones(m, device=DEV) for m, _ in shapes]
        descs = [hiplib.gemm_desc(hiplib.TN, a, b, c, accumulate=True, colsum_out=s) for (a, b), c, s in zip(ops, C, bias)]
        for group in [descs] if grouped else [[d] for d in descs]:
            hiplib.gemm_grouped(group)
        runs.append(C + bias)
    assert all(torch.equal(x, y) for x, y in zip(*runs))


# fp32 tiles of 64x64 and 64x32 whose waves hold four 16x16 accumulators: columns and rows that end in either half of either, every
# operand order and the epilogues that read and write beside the product.  A chain of K multiply-adds errs by at most K eps of the
# terms' sum; what the epilogue adds, a few roundings more.
@pytest.mark.parametrize("layout", ["nt", "nn", "tn"])
@pytest.mark.parametrize("M,N,K", [(2052, 420, 36), (2084, 436, 132), (2112, 404, 64), (2076, 1028, 100)])
def test_f32_tiles_at_their_edges(hiplib, M, N, K, layout):
    lay = getattr(hiplib, layout.upper())
    a, b = torch.randn(M, K, generator=torch.Generator().manual_seed(1)), torch.randn(N, K, generator=torch.Generator().manual_seed(2))
    A, B = (a.t() if layout == "tn" else a).contiguous().to(DEV), (b if layout == "nt" else b.t()).contiguous().to(DEV)
    x, bias = torch.randn(M, N, generator=torch.Generator().manual_seed(3)).to(DEV), torch.randn(N, generator=torch.Generator().manual_seed(4)).to(DEV)
    prod = (a.double() @ b.double().t()).to(DEV)
    bound = (K + 4) * 2.0 ** -24 * ((a.double().abs() @ b.double().abs().t()).to(DEV) + x.double().abs() + bias.double().abs())
    C = torch.full((M, N), float("nan"), device=DEV)
    hiplib.gemm(lay, A, B, C)
    assert bool(((C.double() - prod).abs() <= bound).all())
    C = x.clone()
    hiplib.gemm(lay, A, B, C, accumulate=True)
    assert bool(((C.double() - prod - x.double()).abs() <= bound).all())
    if layout != "tn":
        C = torch.full((M, N), float("nan"), device=DEV)
        hiplib.gemm(lay, A, B, C, bias=bias if layout == "nt" else None, epilogue=hiplib.EPI_RESIDUAL, resid=x)
        want = prod + x.double() + (bias.double() if layout == "nt" else 0)
        assert bool(((C.double() - want).abs() <= bound).all())
    if layout == "nt":
        act, dact = torch.full((M, N), float("nan"), device=DEV), torch.full((M, N), float("nan"), device=DEV)
        hiplib.gemm(lay, A, B, act, bias=bias, epilogue=hiplib.EPI_ACT_DACT, act=hiplib.ACT_RELU, aux_out=dact)
        want = prod + bias.double()
        assert bool(((act.double() - want.clamp(min=0)).abs() <= bound).all()) and bool(((dact == 1) == (act > 0)).all())


# fp32 weight gradients on quarter tiles against the same in a group of too many tiles for them, and each alone: the same bits.
@pytest.mark.parametrize("rows", [132, 196, 260, 1000])
@pytest.mark.parametrize("shapes", [[(384, 128), (128, 512)], [(68, 36), (100, 644), (4, 32)], [(512, 512), (256, 1024)]])
def test_f32_weight_gradients_on_quarter_tiles(hiplib, rows, shapes):
    f32 = lambda *s, seed: torch.randn(*s, generator=torch.Generator().manual_seed(seed)).to(DEV)
    ops = [(f32(rows, m, seed=2 * i), f32(rows, n, seed=2 * i + 1)) for i, (m, n) in enumerate(shapes + [(1024, 768)])]
    outs = []
    for how in ("few", "many", "alone"):
        C = [torch.ones(a.shape[1], b.shape[1], device=DEV) for a, b in ops]
        descs = [hiplib.gemm_desc(hiplib.TN, a, b, c, accumulate=True) for (a, b), c in zip(ops, C)]
        for group in {"few": [descs[:-1]], "many": [descs], "alone": [[d] for d in descs[:-1]]}[how]:
            hiplib.gemm_grouped(group)
        outs.append(C[:-1])
    assert all(torch.equal(a, b) for other in outs[1:] for a, b in zip(outs[0], other))
    for (a, b), c in zip(ops, outs[0]):
        prod, terms = a.double().t() @ b.double(), a.double().abs().t() @ b.double().abs()
        assert bool(((c.double() - 1 - prod).abs() <= (rows + 4) * 2.0 ** -24 * (terms + 1)).all())
