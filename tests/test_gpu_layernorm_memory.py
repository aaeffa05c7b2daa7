"""The decoder layer's memory sqrt(1 - x) beside its LayerNorm: the bits of the separate launches, forward and backward, at row lengths on
either side of what a wave holds, and of where the launches stay separate."""
import pytest
import torch

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("dtype", [torch.bfloat16, torch.float32])
@pytest.mark.parametrize("rows,cols", [(1, 8), (5, 64), (1023, 512), (130, 1032), (33, 2056), (9, 4096),
                                       (7, 1600), (512, 2560), (512, 2568), (513, 3080), (512, 3072), (513, 4096)])
def test_memory(hiplib, dtype, rows, cols):
    g = torch.Generator(device="cuda").manual_seed(rows + cols)
    rand = lambda *shape, t=dtype: torch.randn(*shape, generator=g, device="cuda").to(t)
    x, gain, shift, dy, dres, dm = rand(rows, cols) * 0.3 - 2.0, rand(cols), rand(cols), rand(rows, cols), rand(rows, cols), rand(rows, cols)
    kind, f32 = hiplib.LN_CODES["annotated"], torch.float32
    forward, backward = [], []
    for fused in (False, True):
        y, m = torch.empty_like(x), torch.empty_like(x)
        mean, rinv = torch.empty(rows, device="cuda"), torch.empty(rows, device="cuda")
        hiplib.layernorm_fwd(x, gain, shift, y, mean, rinv, kind, 1e-6, memory=m if fused else None)
        if not fused:
            hiplib.sqrt_one_minus_fwd(x, m)
        dx, dgain, dshift = torch.empty_like(x), torch.zeros(cols, device="cuda", dtype=f32), torch.zeros(cols, device="cuda", dtype=f32)
        partials = torch.empty(hiplib.layernorm_bwd_workspace(cols), device="cuda")
        sums = hiplib.layernorm_bwd_rows(x, gain, mean, rinv, dy, dres, dx, dgain, dshift, partials, kind, 1e-6,
                                         memory=(dm, m) if fused else None)
        hiplib.partial_sums([sums])
        if not fused:
            hiplib.sqrt_one_minus_bwd(dm, m, dx, accumulate=True)
        forward.append((y, m, mean, rinv))
        backward.append((dx, dgain, dshift))
    assert all(torch.equal(a, b) for a, b in zip(*forward))
    assert all(torch.equal(a, b) for a, b in zip(*backward))
    want = torch.sqrt(1.0 - x.double())
    assert float((m.double() - want).norm() / want.norm()) < (3e-3 if dtype == torch.bfloat16 else 3e-7)   # half an ulp of the type
