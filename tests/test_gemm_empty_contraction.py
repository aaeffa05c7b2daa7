"""Products over an empty contraction: no kernel that starts by loading a k-tile may be chosen for them; C is what the epilogue
makes of zeros."""
from ctypes import byref

import pytest
import torch

from bamboo_amd import hip

SHAPES = [(8, 8), (128, 128), (2048, 1000), (4096, 1024), (8192, 4096), (33000, 72), (72, 33000)]     # up to and beyond two 64x64 tiles a CU


def desc(layout, dtype, M, N, A=16, B=16, C=16, c_dtype=None, nb=1):
    d = hip.GemmDesc()
    d.layout, d.dtype, d.c_dtype = layout, dtype, dtype if c_dtype is None else c_dtype
    d.M, d.N, d.K, d.nb1, d.nb2, d.alpha = M, N, 0, 1, nb, 1.0
    d.A, d.B, d.C = A, B, C
    d.lda, d.ldb, d.ldc = (M if layout == hip.TN else 8), (8 if layout == hip.NT else N), N
    return d


@pytest.mark.parametrize("layout", [hip.NT, hip.NN, hip.TN], ids=["nt", "nn", "tn"])
@pytest.mark.parametrize("M,N", SHAPES)
@pytest.mark.parametrize("nb", [1, 48])
def test_no_kernel_that_loads_a_k_tile(layout, M, N, nb):
    assert "wave64x64" in hip.gemm_variant(desc(layout, hip.BF16, M, N, nb=nb))


@pytest.mark.gpu
@pytest.mark.parametrize("dtype", [torch.bfloat16, torch.float32], ids=["bf16", "fp32"])
@pytest.mark.parametrize("layout", ["nt", "nn", "tn"])
@pytest.mark.parametrize("M,N", [(8, 8), (2056, 1000), (4096, 1024)])
def test_epilogue_of_zeros(hiplib, dtype, layout, M, N):
    lay, dev, L = getattr(hip, layout.upper()), "cuda:0", hip.lib()
    some = torch.full((max(M, N), 8), float("nan"), dtype=dtype, device=dev)        # operands: there, but without a column in use
    bias, X = torch.randn(N, device=dev).to(dtype), torch.randn(M, N, device=dev).to(dtype)
    C = torch.full((M, N), float("nan"), dtype=dtype, device=dev)
    d = desc(lay, hip.dtype_code(dtype), M, N, some.data_ptr(), some.data_ptr(), C.data_ptr())
    hip.check(L.bb_gemm(byref(d), hip.stream_ptr()), "bb_gemm")
    assert bool((C == 0).all())
    d.bias, d.epilogue, d.resid = bias.data_ptr(), hip.EPI_RESIDUAL, X.data_ptr()
    hip.check(L.bb_gemm(byref(d), hip.stream_ptr()), "bb_gemm")
    assert torch.equal(C, (bias.float() + X.float()).to(dtype))
    G = torch.randn(M, N, device=dev)
    want = G.clone()
    d = desc(lay, hip.dtype_code(dtype), M, N, some.data_ptr(), some.data_ptr(), G.data_ptr(), hip.F32)
    d.accumulate = 1
    hip.check(L.bb_gemm(byref(d), hip.stream_ptr()), "bb_gemm")
    G2, one, two = G.clone(), d, hip.GemmDesc.from_buffer_copy(d)
    two.C = G2.data_ptr()
    hip.check(L.bb_gemm_grouped((hip.GemmDesc * 2)(one, two), 2, hip.stream_ptr()), "bb_gemm_grouped")
    assert torch.equal(G, want) and torch.equal(G2, want)
