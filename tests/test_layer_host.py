"""What a layer does on the host in a pass: settings changed between passes meet the buffers that the stage was built with, and a
LayerNorm backward makes no tensors on the way (CPU: the kernels are stood in for)."""
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


def test_layernorm_backward_makes_no_tensors(monkeypatch):
    """Issued launch by launch, a LayerNorm backward is host work of a few microseconds: its partial sums lie ready in scratch, each in a
    buffer of its own until the launch that adds them up."""
    from torch.utils._python_dispatch import TorchDispatchMode

    class Ops(TorchDispatchMode):
        seen = 0

        def __torch_dispatch__(self, func, types, args=(), kwargs=None):
            self.seen += 1
            return func(*args, **(kwargs or {}))

    given = []
    monkeypatch.setattr(hip, "layernorm_bwd_rows", lambda *a, **kw: given.append(a[9]))
    layer = TransformerLayer(128, 2, 256)
    layer.w = layer.g = {f"sublayer.{i}.norm.{k}": torch.zeros(128) for i in (0, 1) for k in ("a_2", "b_2")}
    ctx = StageContext(2, 36, torch.bfloat16, "cpu")
    ctx.ensure_scratch(layer.scratch_specs(ctx))
    t, sums = torch.zeros(72, 128), []
    with Ops() as ops:
        for norm in ("sublayer.1.norm", "sublayer.0.norm"):
            layer._layernorm_bwd(sums, ctx, t, norm, t, t, t, t, t)
    assert ops.seen == 0 and given[0].data_ptr() != given[1].data_ptr() and all(g.numel() >= hip.layernorm_bwd_workspace(128) for g in given)
