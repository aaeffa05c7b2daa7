"""The register epilogue's operands at the end of their memory: a residual beside a mask by sign, whose last tile reaches far past the last
row and column.  The operands are the last rows of one allocation of their own size class."""
import pytest
import torch

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("M,N", [(100, 4168), (97, 8200), (2305, 1032), (8200, 1000)])
@pytest.mark.parametrize("layout", ["nt", "nn"])
def test_residual_inside_its_tensor(hiplib, layout, M, N):
    K, lay = 64 if M < 128 else 512, hiplib.NT if layout == "nt" else hiplib.NN
    g = torch.Generator(device="cuda").manual_seed(M)
    rand = lambda *shape: torch.randn(*shape, generator=g, device="cuda").bfloat16()
    A, B, X, R, C = rand(M, K), rand(*((N, K) if layout == "nt" else (K, N))), rand(M, N), rand(M, N), torch.empty(M, N, dtype=torch.bfloat16, device="cuda")
    hiplib.gemm(lay, A, B, C, epilogue=hiplib.EPI_MUL_POS, aux_in=X, resid=R)
    a, b = A.double(), (B.double().t() if layout == "nt" else B.double()).contiguous()
    want = torch.where(X > 0, a @ b + R.double(), 0.0)
    slack = K * 2.0 ** -24 * (a.abs() @ b.abs()) + 2.0 ** -22 * (want.abs() + 8.0)     # fp32 sums, then half an ulp of bf16
    assert ((C.double() - want).abs() <= 2.0 ** -8 * want.abs() + 1.01 * slack).all()
