"""A layer's settings changed between passes meet the buffers that the stage was built with (CPU: the kernels are stood in for)."""
import pytest
import torch

from bamboo_amd import DecoderLayer, TransformerLayer, hip
from bamboo_amd.layers import StageContext

KERNELS = ("gemm_batched", "softmax_fwd", "softmax_bwd", "dropout_apply", "attention_probs_fwd", "attention_probs_bwd")


@pytest.mark.parametrize("forward_only", [False, True], ids=["own lane", "redundant lane"])
@pytest.mark.parametrize("kind", [TransformerLayer, DecoderLayer])
def test_fp32_attention_with_dropout_under_another_activation(monkeypatch, kind, forward_only):
    calls = []
    for name in KERNELS:
        monkeypatch.setattr(hip, name, lambda *a, name=name, **kw: calls.append(name))
    layer = kind(128, 2, 256, activation="gelu_tanh", dropout=0.1)
    layer.layer_idx = 0
    ctx = StageContext(2, 36, torch.float32, "cpu")
    ctx.dropout_base = (1, 2, 3)
    ctx.ensure_scratch(layer.forward_scratch_specs(ctx) if forward_only else layer.scratch_specs(ctx))
    st = {"qkv": torch.zeros(72, 384), "ctx": torch.zeros(72, 128), "prob": torch.zeros(2, 2, 36, 36)}
    kernels = {"gelu_tanh": ["attention_probs_fwd", "attention_probs_bwd"],
               "relu": ["gemm_batched", "softmax_fwd", "dropout_apply", "gemm_batched",
                        "dropout_apply", "gemm_batched", "gemm_batched", "dropout_apply", "softmax_bwd", "gemm_batched", "gemm_batched"]}
    for layer.activation in ("gelu_tanh", "relu", "gelu_tanh"):
        calls.clear()
        layer._attention_fwd(st, ctx)
        if not forward_only:
            layer._attention_bwd(torch.zeros(72, 128), torch.zeros(72, 384), st, ctx)
        want = kernels[layer.activation]
        assert calls == (want[: 1 if layer.activation == "gelu_tanh" else 4] if forward_only else want)
