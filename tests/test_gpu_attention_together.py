"""Attention backward in one launch or two: block counts on either side of a round, sequences around the longest whose row sums a
block keeps, padding that leaves blocks without a key, each head width; against fp64, twice the same bits, without and with dropout."""
import pytest
import torch

from tests import test_gpu_dropout as drop
from tests import test_gpu_kernels as plain

pytestmark = pytest.mark.gpu

SHAPES = [("none", 1, 256, 64, 64), ("none", 1, 257, 64, 64), ("none", 1, 170, 64, 128), ("none", 1, 171, 40, 128), ("none", 2, 256, 33, 32),
          ("none", 1, 2, 2048, 64), ("none", 1, 2, 2049, 64), ("key_padding", 2, 2, 1300, 64), ("causal", 1, 2, 2047, 64), ("causal", 3, 4, 2, 64),
          ("key_padding", 2, 4, 513, 32), ("none", 2, 3, 385, 128),
          # a round and a quarter (128-wide heads: a round), and more
          ("none", 1, 320, 64, 64), ("none", 1, 321, 64, 64), ("none", 1, 168, 64, 128), ("none", 2, 320, 33, 32), ("none", 2, 322, 33, 32),
          ("causal", 1, 576, 65, 64), ("causal", 1, 577, 65, 64)]


@pytest.mark.parametrize("mask,b,a,s,d", SHAPES)
def test_backward(hiplib, mask, b, a, s, d):
    plain.test_fused_attention_fwd_bwd(hiplib, mask, b, a, s, d)


@pytest.mark.parametrize("mask,b,a,s,d", [t for t in SHAPES if t[3] < 2000])
def test_backward_with_dropout(hiplib, mask, b, a, s, d):
    drop.test_fused_attention_dropout_fwd_bwd(hiplib, mask, b, a, s, d)


@pytest.mark.parametrize("mask,b,a,s,d,together", [
    ("causal", 1, 2, 64, 64, True), ("causal", 2, 4, 130, 32, True), ("causal", 1, 2, 300, 128, True), ("causal", 1, 1, 2048, 64, True),
    ("causal", 1, 2, 2049, 64, False), ("causal", 2, 289, 65, 64, False),
    # blocks that are one a CU: a round and a quarter with padding, two and a quarter under a causal mask
    ("key_padding", 2, 8, 640, 64, True), ("key_padding", 2, 8, 641, 64, False), ("causal", 2, 8, 1024, 64, True), ("causal", 1, 9, 1153, 64, False),
    # three heads are on three XCDs
    ("key_padding", 1, 3, 1280, 64, True), ("key_padding", 1, 3, 1281, 64, False), ("causal", 1, 3, 2048, 64, True), ("causal", 2, 288, 65, 64, True),
    ("none", 1, 168, 64, 128, True), ("none", 1, 169, 64, 128, False)])
def test_row_sums(hiplib, mask, b, a, s, d, together):
    """The caller's row sums: left as they were where one launch does both passes, written where the second launch reads them."""
    g = torch.Generator(device="cuda").manual_seed(s)
    qkv, d_out = (torch.randn(b * s, w, generator=g, device="cuda").bfloat16() for w in (3 * a * d, a * d))
    out, lse, delta = torch.empty_like(d_out), torch.empty(b, a, s, device="cuda"), torch.full((b, a, s), -3.0, device="cuda")
    lens = torch.full((b,), s, dtype=torch.int32, device="cuda") if mask == "key_padding" else None
    args = (b, a, s, hiplib.MASK_CODES[mask], lens)
    hiplib.attention_fwd(qkv, out, lse, *args)
    hiplib.attention_bwd(qkv, out, d_out, lse, delta, torch.empty_like(qkv), *args)
    terms = (out.double() * d_out.double()).view(b, s, a, d).transpose(1, 2)
    if together:
        assert (delta == -3.0).all()
    else:       # d products added in fp32, one rounding each
        assert ((delta.double() - terms.sum(-1)).abs() <= d * 2.0 ** -24 * terms.abs().sum(-1)).all()
