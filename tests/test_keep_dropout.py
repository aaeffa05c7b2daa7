"""What a layer with dropout keeps of its attention's decisions (CPU: the memory plan and what the kernels are given)."""
import math

import pytest
import torch

from bamboo_amd import DecoderLayer, TransformerLayer, hip
from bamboo_amd.layers import StageContext
from bamboo_amd.module import PipelineModule

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


def given(monkeypatch):
    calls = []
    for name in ("attention_fwd", "attention_bwd"):
        monkeypatch.setattr(hip, name, lambda *a, name=name, keep=None, **kw: calls.append((name, keep)))
    return calls


@pytest.mark.parametrize("defer", [False, True])
def test_bits_only_for_a_backward_that_reads_them(monkeypatch, defer):
    """A redundant forward, and the backward that comes to its stash after a failover, go without."""
    calls = given(monkeypatch)
    layer = TransformerLayer(128, 2, 256, dropout=0.1)
    layer.layer_idx = 0
    ctx = StageContext(2, 36, torch.bfloat16, "cpu")
    ctx.dropout_base, ctx.defer, ctx.deferred = (1, 2, 3), defer, defer
    ctx.ensure_scratch(layer.scratch_specs(ctx))
    st = {name: torch.zeros(shape, dtype=t) for name, shape, t in layer.stash_specs(ctx)}
    layer._attention_fwd(st, ctx)
    layer._attention_bwd(None, None, st, ctx)
    assert [name for name, _ in calls] == ["attention_fwd", "attention_bwd"]
    assert all(keep is (None if defer else st["keep"]) for _, keep in calls)


def test_first_forward_of_a_checkpointed_group(monkeypatch):
    """What it would leave, the run in front of the group's backward leaves."""
    calls = given(monkeypatch)
    monkeypatch.setattr(hip, "cast", lambda *a, **kw: None)

    class Layer(TransformerLayer):
        def forward(self, x, st, ctx):
            self._attention_fwd(st, ctx)
            return st["out"]

        def backward(self, d_out, d_x, st, ctx):
            self._attention_bwd(None, None, st, ctx)

    ctx = StageContext(2, 36, torch.bfloat16, "cpu")
    ctx.dropout_base = (1, 2, 3)
    layers = [Layer(128, 2, 256, dropout=0.1) for _ in range(3)]
    for i, layer in enumerate(layers):
        layer.layer_idx = i
        ctx.ensure_scratch(layer.scratch_specs(ctx))
    ctx.ensure_scratch([(f"d_layer{i}", (72, 128), torch.bfloat16) for i in (0, 1)])
    module = object.__new__(PipelineModule)
    module.func_buckets, module.activation_checkpoint_interval, module.micro_offset, module.stage_seq = {0: layers}, 2, 0, {0: [36] * 4}
    stash = [{name: torch.zeros(shape, dtype=t) for name, shape, t in layer.stash_specs(ctx)} for layer in layers]
    module._stash, module._kept = {0: [stash]}, {0: [[torch.zeros(72, 128, dtype=torch.bfloat16) for _ in range(3)]]}
    module.forward(torch.zeros(72, 128, dtype=torch.bfloat16), 0, ctx=ctx)
    assert [keep for _, keep in calls] == [None] * 3
    calls.clear()
    module.backward(None, None, 0, ctx=ctx)
    by_layer = [("attention_fwd", 2), ("attention_bwd", 2), ("attention_fwd", 0), ("attention_fwd", 1), ("attention_bwd", 1), ("attention_bwd", 0)]
    assert [name for name, _ in calls] == [name for name, _ in by_layer]
    assert all(keep is stash[i]["keep"] for (_, keep), (_, i) in zip(calls, by_layer))
