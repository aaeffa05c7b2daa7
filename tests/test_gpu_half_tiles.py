"""Small bf16 products whose 64x64 tiles go as two blocks each: rows around half a tile and a tile, the most halves that do and the fewest
that do not, one and several k-tiles; every epilogue kind against fp64, and a long contraction against the same rows among more."""
import pytest
import torch

from tests import test_gpu_direct_epilogue as direct

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("M,N,K,halves", [(1, 64, 64, True), (31, 72, 128, True), (33, 136, 64, True), (64, 128, 576, True), (97, 1000, 192, True),
                                          (1024, 512, 128, True), (1025, 512, 128, False), (100, 4096, 64, True), (100, 4168, 64, False)])
@pytest.mark.parametrize("layout", ["nt", "nn"])
def test_halves(hiplib, layout, M, N, K, halves):
    A, B = torch.empty(M, K, dtype=torch.bfloat16, device="cuda"), torch.empty(*((N, K) if layout == "nt" else (K, N)), dtype=torch.bfloat16, device="cuda")
    variant = hiplib.gemm_variant(hiplib.gemm_desc(hiplib.NT if layout == "nt" else hiplib.NN, A, B, torch.empty(M, N, dtype=torch.bfloat16, device="cuda")))
    assert ("halves_" in variant) == halves
    direct.test_register_epilogue(hiplib, layout, "64x64k64s4", M, N, K)


@pytest.mark.parametrize("layout", ["nt", "nn"])
def test_same_bits_as_whole_tiles(hiplib, layout):
    lay = hiplib.NT if layout == "nt" else hiplib.NN
    g = torch.Generator(device="cuda").manual_seed(3)
    A, B = (torch.randn(*shape, generator=g, device="cuda").bfloat16() for shape in ((1500, 2048), (512, 2048) if layout == "nt" else (2048, 512)))
    few, many = (torch.empty(m, 512, dtype=torch.bfloat16, device="cuda") for m in (700, 1500))
    hiplib.gemm(lay, A[:700], B, few)
    hiplib.gemm(lay, A, B, many)
    assert torch.equal(few, many[:700])
