"""Attention backward whose waves look one sub-tile ahead: lengths around the edges of sub-tiles (32), tiles (64) and blocks, walks of one,
two and three tiles (the ring's stages), padding that ends inside a sub-tile, queries and keys past the end in the last block;
against fp64, twice the same bits, without and with dropout."""
import pytest

from tests import test_gpu_dropout as drop
from tests import test_gpu_kernels as plain

pytestmark = pytest.mark.gpu

SHAPES = [(1, 2, 31, 64), (2, 1, 32, 64), (1, 3, 33, 64), (1, 2, 63, 32), (2, 2, 65, 32), (1, 2, 96, 128), (1, 1, 97, 64), (3, 2, 129, 64),
          (1, 4, 191, 32), (2, 6, 385, 32), (2, 260, 161, 64), (1, 600, 129, 64)]   # the last two beyond a round


@pytest.mark.parametrize("mask", ["none", "causal", "key_padding"])
@pytest.mark.parametrize("b,a,s,d", SHAPES)
def test_walk(hiplib, mask, b, a, s, d):
    plain.test_fused_attention_fwd_bwd(hiplib, mask, b, a, s, d)


@pytest.mark.parametrize("mask", ["none", "causal", "key_padding"])
@pytest.mark.parametrize("b,a,s,d", [t for t in SHAPES if t[0] <= 2 and 63 <= t[2] and t[1] < 100])   # (its key lengths: 37 short of all)
def test_walk_with_dropout(hiplib, mask, b, a, s, d):
    drop.test_fused_attention_dropout_fwd_bwd(hiplib, mask, b, a, s, d)
