"""Replayed launch plans give the bits of passes that are issued launch by launch."""
import pytest
import torch

import bamboo_amd
from bamboo_amd import LayerSpec, PipelineModule, SeededActivationQueue, TransformerLayer

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("first_stage", [False, True], ids=["middle", "first-with-new-data-buffers"])
@pytest.mark.parametrize("dropout,ckpt", [(0.0, 0), (0.1, 0), (0.1, 1)])
def test_replayed_plans_equal_eager_launches(hiplib, dropout, ckpt, first_stage):
    """Four batches with optimizer steps: outputs, sent gradients and weights of an engine that replays its passes (from
    the second batch on, with this batch's dropout keys) and of one whose launch observer keeps it eager.  A first stage
    gets its inputs in other buffers every batch: more variants than the engine remembers."""
    hid, heads, ffn, S, mb, M, seq = 128, 2, 256, 4, 2, 3, 72
    sid = 0 if first_stage else 1

    def make():
        specs = [LayerSpec(TransformerLayer, hid, heads, ffn, activation="gelu_tanh", ln="standard", mask="causal", dropout=dropout)
                 for _ in range(2 * S)]
        model = PipelineModule(specs, num_stages=S, partition_method="uniform", stage_id=sid, dtype=torch.bfloat16, device="cuda:0",
                               activation_checkpoint_interval=ckpt)
        q = SeededActivationQueue((mb, seq, hid), torch.bfloat16, M, stage_ids=[sid, sid + 1], seed=5, device="cuda:0")
        cfg = {"train_micro_batch_size_per_gpu": mb, "gradient_accumulation_steps": M, "bf16": {"enabled": True}}
        engine, _, _, _ = bamboo_amd.initialize(model=model, config=cfg, redundancy_level=1, eager_recovery=True, activation_queue=q,
                                                rc_stream=True, install_signal_handler=False)
        if first_stage:
            engine.set_dataiterator(iter([(q.activations[i % M].clone(), None) for i in range(6 * M)]))
        return engine, q
    (eager, q0), (replay, q1) = make(), make()
    eager.set_gemm_hook(lambda desc, launch, stream: launch())
    for _ in range(6):
        eager.train_batch()
        replay.train_batch()
        torch.cuda.synchronize()
        for key, t in q0.sent.items():
            assert torch.equal(t, q1.sent[key]), key
        for key, t in q0.sent_grads.items():
            assert torch.equal(t, q1.sent_grads[key]), key
    assert torch.equal(eager.module.stage_params[sid].master, replay.module.stage_params[sid].master)
    assert not eager._plans and len(replay._plans) == 3 * M
    assert all(1 <= len(v) <= replay.PLAN_VARIANTS for v in replay._plans.values())
    assert eager.module.micro_offset == replay.module.micro_offset
