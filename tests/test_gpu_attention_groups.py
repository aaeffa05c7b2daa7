"""Attention whose walk over the tiles is shared by groups of waves (masked, few blocks), where that can go wrong: lengths around
the rules' limits and the tiles' edges, fewer tiles than groups in front of the causal diagonal, each head width in each
shape of a block; against fp64, twice the same bits, without and with dropout."""
import pytest

from tests import test_gpu_dropout as drop
from tests import test_gpu_kernels as plain

pytestmark = pytest.mark.gpu

# waves x groups of a block, forward and backward (4x1: the walk is not shared)
SHAPES = [(1, 2, 160, 64), (2, 3, 193, 64),                             # 2x4, 2x1
          (1, 5, 321, 64),                                              # 2x4, 2x4 in one launch
          (1, 2, 2100, 64),                                             # 2x4, 2x4 in two
          (2, 8, 520, 64), (1, 22, 450, 64),                            # 2x4, 2x2 in one; with padding the second in two
          (2, 17, 225, 64),                                             # 2x4, 2x2 if causal, else 2x1
          (1, 11, 641, 64), (1, 9, 1210, 64),                           # 2x4, 2x2 or with dropout 2x4, 2x4
          (1, 36, 448, 64), (1, 43, 577, 64),                           # 2x2, 4x1
          (1, 11, 1537, 64),                                            # 2x2, 4x2
          (1, 33, 1025, 64),                                            # 2x2 if causal, else 4x1, both backward 4x1
          (1, 4, 80, 32), (2, 60, 289, 32),                             # pairs of heads: 2x1
          (2, 6, 257, 32), (2, 16, 600, 32), (2, 16, 650, 32),          # 2x2, with padding the last in two launches
          (1, 2, 448, 128), (2, 4, 521, 128), (1, 30, 500, 128),        # 4x2, with padding the last in two
          (1, 38, 500, 128)]                                            # in two


@pytest.mark.parametrize("mask", ["causal", "key_padding"])
@pytest.mark.parametrize("b,a,s,d", SHAPES)
def test_shared_walk(hiplib, mask, b, a, s, d):
    plain.test_fused_attention_fwd_bwd(hiplib, mask, b, a, s, d)


@pytest.mark.parametrize("mask", ["causal", "key_padding"])
@pytest.mark.parametrize("b,a,s,d", SHAPES)
def test_shared_walk_with_dropout(hiplib, mask, b, a, s, d):
    drop.test_fused_attention_dropout_fwd_bwd(hiplib, mask, b, a, s, d)
