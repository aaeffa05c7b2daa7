"""A stage whose attention keeps its dropout decisions against one that makes them again: the same bits in every result, on the full and
on a checkpointed stash, beside redundant forwards and after a failover onto their stash."""
import pytest
import torch

import bamboo_amd
from bamboo_amd import DecoderLayer, LayerSpec, PipelineModule, SeededActivationQueue, TransformerLayer

pytestmark = pytest.mark.gpu


def batches(kind, keep, ckpt):
    hid, heads, ffn, S, sid, mb, seq, M = 128, 2, 256, 4, 1, 2, 96, 3
    specs = [LayerSpec(kind, hid, heads, ffn, dropout=0.1, keep_dropout=keep) for _ in range(2 * S)]
    model = PipelineModule(specs, num_stages=S, partition_method="uniform", stage_id=sid, dtype=torch.bfloat16, device="cuda:0", base_seed=99,
                           activation_checkpoint_interval=ckpt)
    queue = SeededActivationQueue((mb, seq, hid), torch.bfloat16, M, stage_ids=[sid, sid + 1], seed=5, device="cuda:0")
    queue.activations = [a * 0.3 - 2.0 for a in queue.activations]       # (the decoder's memory is defined below 1)
    config = {"train_micro_batch_size_per_gpu": mb, "gradient_accumulation_steps": M, "optimizer": {"type": "Adam", "params": {"lr": 1e-3}},
              "bf16": {"enabled": True}}
    engine, _, _, _ = bamboo_amd.initialize(model=model, config=config, redundancy_level=1, eager_recovery=True, activation_queue=queue,
                                            install_signal_handler=False)
    for _ in range(2):
        engine.train_batch()
    return model, [engine.module.stage_params[sid].master.clone(), *(queue.sent_grads[k].clone() for k in sorted(queue.sent_grads))]


@pytest.mark.parametrize("ckpt", [0, 1, 2])
@pytest.mark.parametrize("kind", [TransformerLayer, DecoderLayer])
def test_same_results(hiplib, kind, ckpt):
    model, kept = batches(kind, True, ckpt)
    assert "keep" in model._stash[1][0][0]
    model, made = batches(kind, False, ckpt)
    assert "keep" not in model._stash[1][0][0]
    assert len(kept) > 1 and all(torch.equal(a, b) for a, b in zip(kept, made)) and all(torch.isfinite(a).all() for a in kept)


@pytest.mark.parametrize("kind", [TransformerLayer, DecoderLayer])
def test_backward_of_a_deferred_forward(hiplib, kind):
    """The forward of a redundant pass and the backward that follows a failover on its stash, against the normal pair."""
    model, _ = batches(kind, True, 0)
    sid, ctx = 1, model.prepare_context([1], 2, 96)
    g = torch.Generator(device="cuda:0").manual_seed(1)
    x, d = (torch.randn(192, 128, generator=g, device="cuda:0") * 0.3 - 2.0).bfloat16(), torch.randn(192, 128, generator=g, device="cuda:0").bfloat16()
    results = []
    for defer in (False, True):
        ctx.dropout_base = (99, 7, 1)
        for st in model._stash[sid][0]:
            for name in ("keep", "keep_src"):
                if name in st:
                    st[name].fill_(0x55555555 if defer else 0)           # neither written nor read
        model.stage_params[sid].grad.zero_()
        out = model.forward(x, sid, slot=0, ctx=ctx, defer=defer).clone()
        if defer:
            assert all((st[name] == 0x55555555).all() for st in model._stash[sid][0] for name in ("keep", "keep_src") if name in st)
        dx = model.backward(d, torch.empty_like(x), sid, slot=0, ctx=ctx, deferred=defer)
        results.append((out, dx, model.stage_params[sid].grad.clone()))
    assert all(torch.equal(a, b) for a, b in zip(*results))
