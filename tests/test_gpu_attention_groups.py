"""Attention whose walk over the tiles is shared by groups of waves (masked, few blocks), where that can go wrong: lengths around
the rules' limits and the tiles' edges, fewer tiles than groups in front of the causal diagonal, each head width in each
shape of a block; against fp64, twice the same bits, without and with dropout."""
import pytest

from tests import test_gpu_dropout as drop
from tests import test_gpu_kernels as plain

pytestmark = pytest.mark.gpu

SHAPES = [(1, 2, 160, 64), (2, 3, 193, 64), (1, 5, 321, 64), (1, 4, 80, 32), (2, 6, 257, 32),                # two waves in four groups
          (1, 36, 448, 64), (1, 43, 577, 64), (2, 60, 289, 32), (1, 2, 448, 128), (2, 4, 521, 128)]          # four waves in two


@pytest.mark.parametrize("mask", ["causal", "key_padding"])
@pytest.mark.parametrize("b,a,s,d", SHAPES)
def test_shared_walk(hiplib, mask, b, a, s, d):
    plain.test_fused_attention_fwd_bwd(hiplib, mask, b, a, s, d)


@pytest.mark.parametrize("mask", ["causal", "key_padding"])
@pytest.mark.parametrize("b,a,s,d", SHAPES)
def test_shared_walk_with_dropout(hiplib, mask, b, a, s, d):
    drop.test_fused_attention_dropout_fwd_bwd(hiplib, mask, b, a, s, d)
