"""Replayed launch plans give the bits of passes that are issued launch by launch."""
import pytest
import torch

import bamboo_amd
from bamboo_amd import (BottleNeck, DecoderLayer, FinalLayerNorm, LayerSpec, MSELoss, PipelineModule, SeededActivationQueue, SumLast,
                        TransformerLayer, hip)

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("first_stage", [False, True], ids=["middle", "first-with-new-data-buffers"])
@pytest.mark.parametrize("dropout,ckpt", [(0.0, 0), (0.1, 0), (0.1, 1)])
def test_replayed_plans_equal_eager_launches(hiplib, dropout, ckpt, first_stage):
    """Four batches with optimizer steps: outputs, sent gradients and weights of an engine that replays its passes (from
    the second batch on, with this batch's dropout keys) and of one whose launch observer keeps it eager.  A first stage
    gets its inputs in other buffers every batch."""
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


class MovingQueue(SeededActivationQueue):
    """Hands out the same values in other buffers at every call."""

    def __init__(self, *a, **kw):
        self.handed = []
        super().__init__(*a, **kw)

    def _moved(self, t):
        self.handed.append(t.clone())      # kept: the next clone lies elsewhere
        return self.handed[-1]

    def recv_activation(self, k):
        return self._moved(super().recv_activation(k))

    def recv_grad(self, k, stage_id):
        return self._moved(super().recv_grad(k, stage_id))

    def key_len(self, k):
        return None if self.key_lens is None else self._moved(super().key_len(k))


class BubbleQueue(MovingQueue):
    """Nothing arrives while redundant forwards are pending: they go out one layer at a time."""

    engine = None

    def activation_arrived(self, k):
        return not self.engine._rc_pending

    def grad_arrived(self, k, stage_id):
        return not self.engine._rc_pending


S, M = 4, 3


def layers(kind, n=2):
    """(specs of S stages of n layers, activation shape, output shape, stage whose passes run, further options)"""
    enc = dict(activation="gelu_tanh", ln="standard", mask="key_padding", dropout=0.1)
    script = dict(activation="relu", ln="annotated", mask="none", dropout=0.1)
    if kind == "decoder":
        return [LayerSpec(DecoderLayer, 64, 2, 128, **script) for _ in range(n * S)], (2, 40, 64), 1, {}
    if kind == "resnet":
        blocks = [(64, 16, 1)] * n + [(64, 32, 2)] + [(128, 32, 1)] * (3 * n - 1)
        sides = [8] * (n + 1) + [4] * (3 * n - 1)
        specs = [LayerSpec(BottleNeck, ci, cm, stride=st, height=s, width=s) for (ci, cm, st), s in zip(blocks, sides)]
        return specs, (3, 64, 64), 1, dict(out_shapes={1: (3, 16, 128), 2: (3, 16, 128)})
    if kind == "resnet_wide":    # the implicit convolutions, the strip sums in the epilogues, gradients masked by the block behind
        specs = [LayerSpec(BottleNeck, 256, 64, height=14, width=14) for _ in range(n * S)]
        return specs, (2, 196, 256), 1, {}
    if kind == "tail":
        specs = [LayerSpec(TransformerLayer, 64, 2, 128, **script) for _ in range(n * S)]
        return specs + [LayerSpec(FinalLayerNorm, 64, ln="annotated"), LayerSpec(SumLast, 64)], (2, 40, 64), S - 1, {}
    return [LayerSpec(TransformerLayer, 64, 2, 128, **enc) for _ in range(n * S)], (2, 40, 64), 1, dict(key_len_range=(9, 40))


def make_engine(kind, queue=SeededActivationQueue, dtype=torch.bfloat16, ckpt=0, n=2, rc=True, **kw):
    specs, shape, sid, options = layers(kind, n)
    tail = kind == "tail"
    parts = [i * n for i in range(S)] + [len(specs)]
    model = PipelineModule(specs, num_stages=S, partition_method="custom", custom_partitions=parts, stage_id=sid, dtype=dtype, device="cuda:0",
                           loss_fn=MSELoss() if tail else None, activation_checkpoint_interval=ckpt)
    rc = rc and not tail
    q = queue(shape, dtype, M, stage_ids=[sid] + [sid + 1] * rc, seed=5, device="cuda:0", **options)
    if kind == "decoder":
        q.activations = [t * 0.5 - 4 for t in q.activations]     # defined for inputs below 1
    cfg = {"train_micro_batch_size_per_gpu": shape[0], "gradient_accumulation_steps": M, "bf16": {"enabled": dtype == torch.bfloat16},
           "optimizer": {"type": "Adam", "params": {"lr": 1e-3}}}
    engine, _, _, _ = bamboo_amd.initialize(model=model, config=cfg, redundancy_level=int(rc), eager_recovery=rc, activation_queue=q,
                                            install_signal_handler=False, **kw)
    if tail:
        g = torch.Generator().manual_seed(9)
        engine.set_dataiterator(iter([(None, torch.randn(shape[0], shape[1], generator=g)) for _ in range(12 * M)]))
    return engine, q


def eager(engine):
    engine.set_gemm_hook(lambda desc, launch, stream: launch())     # a launch observer keeps an engine from replaying


def assert_same_state(a, b):
    """Weights, moments and running statistics of two engines, what they sent and their losses, bit for bit."""
    for sid, sp in a.module.stage_params.items():
        other = b.module.stage_params[sid]
        for arena in ("master", "compute", "exp_avg", "exp_avg_sq"):
            assert torch.equal(getattr(sp, arena), getattr(other, arena)), (sid, arena)
        for la, lb in zip(sp.layers, other.layers):
            for i, stats in (getattr(la, "running", None) or {}).items():
                assert all(torch.equal(x, y) for x, y in zip(stats, lb.running[i])), (sid, i)
    for sent in ("sent", "sent_grads"):
        x, y = getattr(a.queue, sent), getattr(b.queue, sent)
        assert x.keys() == y.keys() and all(torch.equal(x[k], y[k]) for k in x), sent
    assert torch.equal(a.agg_train_loss, b.agg_train_loss) and a.module.micro_offset == b.module.micro_offset


@pytest.mark.parametrize("kind,dtype,kw", [
    ("encoder", torch.bfloat16, dict(rc_stream=True, rc_issue="bubble")), ("encoder", torch.bfloat16, dict(ckpt=1)),
    ("encoder", torch.float32, {}), ("decoder", torch.bfloat16, dict(rc_stream=True)), ("decoder", torch.float32, {}),
    ("resnet", torch.bfloat16, dict(rc_stream=True)), ("resnet", torch.float32, {}), ("resnet_wide", torch.bfloat16, {}),
    ("resnet_wide", torch.bfloat16, dict(ckpt=2)), ("tail", torch.bfloat16, {})])
def test_replays_take_other_buffers(hiplib, kind, dtype, kw):
    """Inputs, received gradients and key lengths in new buffers at every call: every layer kind, running statistics, a last
    stage, redundant forwards issued layer by layer.  Nothing is recorded after the first batch."""
    bubble = kw.get("rc_issue") == "bubble"
    (a, _), (b, q) = make_engine(kind, dtype=dtype, **kw), make_engine(kind, BubbleQueue if bubble else MovingQueue, dtype=dtype, **kw)
    eager(a)
    q.engine = b
    counts = []
    for _ in range(4):
        a.train_batch()
        b.train_batch()
        torch.cuda.synchronize()
        assert_same_state(a, b)
        counts.append((len(b._plans), sum(len(v) for v in b._plans.values())))
    assert counts[0] == counts[-1] and counts[0][0] == counts[0][1] > 0 and not a._plans
    assert bubble == any(slot[0] == "F1" for slot in b._plans)


@pytest.mark.parametrize("rc_issue", ["reference", "bubble"])
@pytest.mark.parametrize("kind", ["encoder", "resnet"])
def test_failover_after_replayed_batches(hiplib, kind, rc_issue):
    """The successor is lost in the fourth batch: the promoted stage's passes, and the batches after it, equal the eager ones."""
    kw = dict(rc_stream=True, rc_issue=rc_issue)
    (a, qa), (b, qb) = make_engine(kind, **kw), make_engine(kind, MovingQueue, **kw)
    eager(a)
    for batch in range(6):
        if batch == 3:
            qa.preempt_successor(1, 1)
            qb.preempt_successor(1, 1)
        a.train_batch()
        b.train_batch()
        torch.cuda.synchronize()
        assert_same_state(a, b)
    assert b.stage_ids == [1, 2] and b._plans


def refused(engine):
    """The batch is refused by a check on the host."""
    with pytest.raises(hip.HipKernelError):
        engine.train_batch()
    torch.cuda.synchronize()
    engine._clean_pipe_buffers()


@pytest.mark.parametrize("kind", ["encoder", "resnet"])
def test_a_wrong_operand_on_a_later_batch_is_refused(hiplib, kind):
    """A short micro-batch, another type or stride in a place that the recorded passes know."""
    engine, q = make_engine(kind)
    for _ in range(3):
        engine.train_batch()
    x, g = q.activations[1], q.grads[1][2]
    for bad in (x[:1], x.float().to(torch.float16), x.transpose(0, 1).contiguous().transpose(0, 1)[:1]):
        q.activations[1] = bad
        refused(engine)
    q.activations[1] = x
    q.grads[1][2] = g[:1]
    refused(engine)
    q.grads[1][2] = g
    if kind == "encoder":
        n = q.key_lens[0]
        q.key_lens[0] = n.long()
        refused(engine)
        q.key_lens[0] = n
    engine.train_batch()


SETTINGS = [("encoder", "dropout", 0.0), ("encoder", "dropout", 0.25), ("encoder", "mask", "causal"), ("encoder", "eps", 1e-2), ("encoder", "base_seed", 77),
            ("resnet", "momentum", 0.5), ("resnet", "eps", 1e-1), ("resnet", "running", None), ("tail", "dropout", 0.0)]


@pytest.mark.parametrize("kind,name,value", SETTINGS)
def test_settings_changed_between_batches_take_effect(hiplib, kind, name, value):
    """As in an engine that replays nothing: the next batch runs with the new setting, in every layer."""
    (a, _), (b, _) = make_engine(kind, replay=False), make_engine(kind)
    for batch in range(5):
        if batch == 2:
            for engine in (a, b):
                for sid in engine.module.func_buckets:
                    for obj in [engine.module] if name == "base_seed" else engine.module.func_buckets[sid]:
                        if hasattr(obj, name):
                            setattr(obj, name, value)
        a.train_batch()
        b.train_batch()
        torch.cuda.synchronize()
        assert_same_state(a, b)
    assert b._plans and not a._plans
