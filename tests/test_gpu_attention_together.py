"""Attention backward in one launch or two: block counts on either side of a round, sequences around the longest whose row sums a
block keeps, padding that leaves blocks without a key, each head width; against fp64, twice the same bits, without and with dropout."""
import pytest

from tests import test_gpu_dropout as drop
from tests import test_gpu_kernels as plain

pytestmark = pytest.mark.gpu

SHAPES = [("none", 1, 256, 64, 64), ("none", 1, 257, 64, 64), ("none", 1, 170, 64, 128), ("none", 1, 171, 40, 128), ("none", 2, 256, 33, 32),
          ("none", 1, 2, 2048, 64), ("none", 1, 2, 2049, 64), ("key_padding", 2, 2, 1300, 64), ("causal", 1, 2, 2047, 64), ("causal", 3, 4, 2, 64),
          ("key_padding", 2, 4, 513, 32), ("none", 2, 3, 385, 128)]


@pytest.mark.parametrize("mask,b,a,s,d", SHAPES)
def test_backward(hiplib, mask, b, a, s, d):
    plain.test_fused_attention_fwd_bwd(hiplib, mask, b, a, s, d)


@pytest.mark.parametrize("mask,b,a,s,d", [t for t in SHAPES if t[3] < 2000])
def test_backward_with_dropout(hiplib, mask, b, a, s, d):
    drop.test_fused_attention_dropout_fwd_bwd(hiplib, mask, b, a, s, d)
