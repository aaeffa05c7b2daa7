"""The squared-error head over few values, in one block: fewer than one a thread, several, the most it takes and one more; against fp64."""
import pytest
import torch

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("dtype", [torch.bfloat16, torch.float32])
@pytest.mark.parametrize("n", [1, 63, 1024, 1025, 3000, 4096, 4097])
def test_mse_of_few_values(hiplib, dtype, n):
    g = torch.Generator(device="cuda").manual_seed(n)
    y, t = (torch.randn(n, generator=g, device="cuda").to(dtype) for _ in range(2))
    loss, ws = torch.full((1,), 2.0, device="cuda"), torch.empty(hiplib.mse_workspace(), device="cuda")
    d = y.double() - t.double()
    for accumulate, start in ((True, 2.0), (False, 0.0)):
        dy = torch.empty_like(y)
        hiplib.mse_fwd_bwd(y, t, dy, 0.5, loss, accumulate, ws)
        want = start + float((d * d).mean())
        assert abs(float(loss) - want) <= 4e-6 * want      # at most 24 fp32 roundings of sums of positive terms
        assert torch.allclose(dy.double(), 0.5 * 2 * d / n, rtol=2.0 ** -8 if dtype == torch.bfloat16 else 1e-6, atol=0)
