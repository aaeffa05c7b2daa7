"""What a layer with dropout keeps of its attention's decisions (CPU: the memory plan and what the kernels are given)."""
import math

import pytest
import torch

from bamboo_amd import DecoderLayer, TransformerLayer
from bamboo_amd.layers import StageContext

kinds = pytest.mark.parametrize("kind", [TransformerLayer, DecoderLayer])


def stash(layer, batch, seq, dtype=torch.bfloat16):
    specs = {name: (shape, t) for name, shape, t in layer.stash_specs(StageContext(batch, seq, dtype, "cpu"))}
    return specs, sum(math.prod(shape) * t.itemsize for shape, t in specs.values())


@kinds
@pytest.mark.parametrize("heads,head_dim", [(25, 64), (16, 32), (8, 128)])
def test_memory_is_linear_in_the_length(kind, heads, head_dim):
    hidden = heads * head_dim
    layer, plain = (kind(hidden, heads, 4 * hidden, dropout=p) for p in (0.1, 0.0))
    attentions = 2 if kind is DecoderLayer else 1
    for seq in (1, 33, 175, 1024, 32 * head_dim - 5, 32 * head_dim, 32 * head_dim + 1, 32768):
        specs, total = stash(layer, 2, seq)
        extra = total - stash(plain, 2, seq)[1]
        assert 0 <= extra <= attentions * 2 * 2 * ((seq + 63) // 64 * 64 * hidden * 2)      # two [rows, hidden] tensors of bf16 for each
        if seq > 32 * head_dim:
            assert extra == 0
        else:
            assert "keep" in specs and (seq % 64 or extra == attentions * 2 * heads * seq * seq // 8)


@kinds
def test_caller_may_decline(kind):
    layer = kind(1024, 16, 4096, dropout=0.1, keep_dropout=False)
    assert stash(layer, 8, 1024) == stash(kind(1024, 16, 4096), 8, 1024)
    layer.keep_dropout = True
    assert {"keep"} <= stash(layer, 8, 1024)[0].keys() and "keep" not in stash(layer, 8, 1024, torch.float32)[0]
