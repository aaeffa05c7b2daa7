"""The batches whose speed this framework is judged by: what a user of ``PipelineEngine.train_batch`` has it do.

A case is one pipeline stage (1F1B stream over ``M`` micro-batches: own forward and backward passes, the redundant
forwards of the stage it shadows, one fused Adam step), built the way a program builds it: ``PipelineModule`` over layer
specs, ``bamboo_amd.initialize``, one ``train_batch()`` per pass.  Shapes, variants and options are those of the
benchmark's configurations, of the reference scripts' layers and of the stages the tests run, at full and at small sizes.

Fields: ``kind`` (encoder, decoder, tail, resnet), ``dtype``, sizes, ``M`` micro-batches; ``rc`` redundant forwards of
an equally deep shadow stage (``rc_stream``: on a second stream), ``ckpt`` activation-checkpoint interval, ``clip``
gradient clipping (global norm, 0 = off).
"""
import gc
import itertools
import math

import torch

import bamboo_amd
from bamboo_amd import (BottleNeck, DecoderLayer, FinalLayerNorm, LayerSpec, MSELoss, PipelineModule, SeededActivationQueue,
                        SumLast, TransformerLayer)

GPT = dict(activation="gelu_tanh", ln="standard", mask="causal")
BERT = dict(activation="gelu_tanh", ln="standard", mask="key_padding")
SCRIPT = dict(activation="relu", ln="annotated", mask="none")   # the reference's transformer and GPT-2 scripts
STAGES = 4                                                      # pipeline depth; stage 1 is the one that runs here
FLOP_CAP, BYTE_CAP = 3.3e13, 6e9                                # a drawn case stays below the largest listed one


def _encoder(name, dtype, heads, head_dim, ffn, layers, seq, mb, M, variant, kind="encoder", dropout=0.0, rc=1, rc_stream=1,
             ckpt=0, clip=0.0):
    return dict(name=name, kind=kind, dtype=dtype, heads=heads, hidden=heads * head_dim, ffn=ffn, layers=layers, seq=seq, mb=mb,
                M=M, dropout=dropout, rc=rc, rc_stream=rc_stream, ckpt=ckpt, clip=clip, **variant)


def _resnet(name, dtype, mid, side, layers, mb, M, stride=1, rc=1, rc_stream=1):
    return dict(name=name, kind="resnet", dtype=dtype, mid=mid, side=side, layers=layers, mb=mb, M=M, stride=stride, rc=rc,
                rc_stream=rc_stream, ckpt=0, clip=0.0)


def listed():
    return [
        # a toy stage, as the smoke run and most tests have it: launches and host work are all there is
        _encoder("toy_bf16", "bf16", 2, 64, 256, 1, 64, 2, 4, GPT, rc_stream=0),
        # the same at fp32 with the reference script's layers
        _encoder("toy_fp32", "fp32", 2, 64, 256, 2, 64, 2, 4, SCRIPT, rc_stream=0),
        # the GPT-2 script's decoder layers at its default width (512 / 16 heads) and dropout
        _encoder("script_decoder", "bf16", 16, 32, 2048, 2, 128, 8, 4, SCRIPT, kind="decoder", dropout=0.1),
        # the transformer script's last stage (final LayerNorm, sum, MSE), gradient clipping, an odd sequence length
        _encoder("script_tail_odd", "bf16", 8, 64, 2048, 3, 175, 6, 4, SCRIPT, kind="tail", rc=0, rc_stream=0, clip=1.0),
        # GPT-2-small in fp32: the correctness configuration
        _encoder("gpt2_small_fp32", "fp32", 12, 64, 3072, 2, 512, 4, 8, GPT),
        # GPT-2-medium, the benchmark's headline stage
        _encoder("gpt2_medium", "bf16", 16, 64, 4096, 6, 1024, 8, 4, GPT),
        # the same width as the reference scripts train it: ReLU, annotated LayerNorm, no mask, dropout 0.1, no redundancy
        _encoder("script_medium_dropout", "bf16", 16, 64, 4096, 4, 1024, 8, 4, SCRIPT, dropout=0.1, rc=0, rc_stream=0),
        # BERT-large with ragged key lengths
        _encoder("bert_large", "bf16", 16, 64, 4096, 4, 512, 16, 4, BERT),
        # GPT-2-1.5B: 25 heads, 1600 columns; the largest
        _encoder("gpt2_xl", "bf16", 25, 64, 6400, 8, 1024, 4, 4, GPT),
        # a long, odd sequence at small batch, redundant forwards on the own stream, checkpointed activations
        _encoder("long_odd_ckpt", "bf16", 12, 64, 3072, 4, 2043, 1, 4, BERT, rc_stream=0, ckpt=1),
        # ResNet-152 conv4_x blocks
        _resnet("resnet152_conv4", "bf16", 256, 14, 12, 32, 4),
        # a down-sampling ResNet stage (28x28 -> 14x14, projection shortcut) at a smaller batch
        _resnet("resnet_down", "bf16", 256, 28, 3, 16, 4, stride=2),
    ]


def draw(rng):
    log = lambda lo, hi: math.exp(rng.uniform(math.log(lo), math.log(hi)))
    while True:
        kind = rng.choice(["encoder"] * 6 + ["decoder", "tail", "resnet", "resnet"])
        dtype = "fp32" if rng.random() < 0.2 else "bf16"
        rc = 0 if kind == "tail" else int(rng.random() < 0.7)
        rc_stream = int(rc and rng.random() < 0.6)
        M = rng.choice([2, 3, 4, 6, 8])
        mb = round(log(1, 16))
        if kind == "resnet":
            stride = 2 if rng.random() < 0.3 else 1
            side = rng.randint(8, 28)
            c = _resnet("", dtype, rng.choice([64, 128, 256]), side, rng.randint(2, 8), max(4, 2 * mb), M, stride, rc, rc_stream)
        else:
            seq = round(log(33, 2048))
            head_dim, heads = rng.choice([64, 64, 64, 64, 32, 128]), round(log(2, 25))
            heads = max(2, heads // 2 * 2) if head_dim == 32 else max(2, heads // 2) if head_dim == 128 else heads
            if dtype == "fp32":          # scores are kept: rows of whole 16-byte vectors, moderate lengths
                seq = max(36, min(seq, 512) // 4 * 4)
            variant = SCRIPT if kind in ("decoder", "tail") else rng.choice([GPT, GPT, BERT, SCRIPT])
            dropout = 0.1 if rng.random() < 0.3 else 0.0
            ckpt = int(kind == "encoder" and rng.random() < 0.15)
            layers = rng.randint(1, 6)
            if kind == "decoder":        # two sublayers more per layer, and its memory wants inputs that stay below 1
                heads, layers = max(2, min(heads, 1024 // head_dim)), (layers + 2) // 3
            c = _encoder("", dtype, heads, head_dim, rng.choice([2, 4, 4]) * heads * head_dim, layers, seq, mb, M, variant,
                         kind=kind, dropout=dropout, rc=rc, rc_stream=rc_stream, ckpt=ckpt, clip=float(rng.random() < 0.25))
        del c["name"]
        w = work(c)
        if w["flops"] <= FLOP_CAP * (0.05 if dtype == "fp32" else 1.0) and w["bytes"] <= BYTE_CAP:
            return c


# ------------------------------------------------------------------------------------------------ a program's set-up
# layers whose weights arrive from elsewhere: no random host-side initialisation, see _load
class _Encoder(TransformerLayer):
    def init_params(self, master, seed):
        pass


class _Decoder(DecoderLayer):
    def init_params(self, master, seed):
        pass


class _Block(BottleNeck):
    def init_params(self, master, seed):
        pass


class _Queue(SeededActivationQueue):
    """The neighbours' tensors, generated on the GPU; keeps the redundant outputs of the last batch at hand."""

    pipe_buffers = None
    scale, shift = 1.0, 0.0
    redundant = ()

    def _randn(self, tag, shape=None):
        g = torch.Generator(device=self.device).manual_seed(self._tag_seed(tag))
        t = torch.randn(shape or self.shape, generator=g, dtype=torch.float32, device=self.device)
        if tag[0] == "act":
            t = t * self.scale + self.shift
        return t.to(self.dtype)

    def end_batch(self, stage_ids):
        self.redundant = [t for key, bufs in self.pipe_buffers().items() for t in bufs
                          if key.startswith("output_") and int(key[7:]) not in stage_ids and t is not None]


class _DecoderQueue(_Queue):
    scale, shift = 0.5, -4.0   # the script's decoder layers are defined for inputs below 1


def _load(sp, seed, std):
    """Weights of a trained-like model: N(0, std) (He-normal for convolutions), norms near one, small biases."""
    g = torch.Generator(device=sp.device).manual_seed(seed)
    sp.master.normal_(0.0, std, generator=g)
    for key, t in sp.named(sp.master).items():
        if t.dim() == 1:
            gain = key.endswith("a_2") or ("residual_function" in key or "shortcut" in key) and key.endswith("weight")
            t.add_(1.0 if gain else 0.0)
        elif "residual_function" in key or "shortcut" in key:
            t.mul_(1.0 / std * math.sqrt(2.0 / (t.numel() // t.shape[0])))
    sp.refresh_compute()


def _resnet_blocks(case):
    """(in, mid, stride) of every block of the four stages, the image side in front of each, for a stage that may halve it."""
    mid, n, s = case["mid"], case["layers"], case["stride"]
    first = (2 * mid, mid, 2) if s == 2 else (4 * mid, mid, 1)
    before = (first[0], first[0] // 4, 1)
    blocks = [before] * n + [first] + [(4 * mid, mid, 1)] * (3 * n - 1)
    small = (case["side"] - 1) // s + 1
    return blocks, [case["side"]] * (n + 1) + [small] * (3 * n - 1), small


def prepare(case, seed):
    gc.collect()     # an engine is part of reference cycles: the previous one's memory comes back first
    dtype = torch.bfloat16 if case["dtype"] == "bf16" else torch.float32
    mb, M, n, kind = case["mb"], case["M"], case["layers"], case["kind"]
    stage, loss, data, out_shapes, parts = 1, None, None, None, [i * n for i in range(STAGES + 1)]
    if kind == "resnet":
        blocks, sides, small = _resnet_blocks(case)
        specs = [LayerSpec(_Block, ci, cm, stride=st, height=side, width=side) for (ci, cm, st), side in zip(blocks, sides)]
        shape = (mb, case["side"] ** 2, blocks[n][0])
        out_shapes = {s: (mb, small * small, 4 * case["mid"]) for s in (1, 2)}
    else:
        layer = _Decoder if kind == "decoder" else _Encoder
        specs = [LayerSpec(layer, case["hidden"], case["heads"], case["ffn"], activation=case["activation"], ln=case["ln"],
                           mask=case["mask"], dropout=case["dropout"]) for _ in range(n * STAGES)]
        shape = (mb, case["seq"], case["hidden"])
        if kind == "tail":
            specs += [LayerSpec(FinalLayerNorm, case["hidden"], ln=case["ln"]), LayerSpec(SumLast, case["hidden"])]
            stage, loss, parts[-1] = STAGES - 1, MSELoss(), n * STAGES + 2
    model = PipelineModule(specs, num_stages=STAGES, partition_method="custom", custom_partitions=parts, stage_id=stage, dtype=dtype,
                           device="cuda:0", loss_fn=loss, activation_checkpoint_interval=case["ckpt"])
    key_lens = (max(1, case["seq"] // 4), case["seq"]) if case.get("mask") == "key_padding" else None
    queue = (_DecoderQueue if kind == "decoder" else _Queue)(
        shape, dtype, M, stage_ids=[stage] if kind == "tail" or not case["rc"] else [1, 2], seed=seed, grad_mode="queue",
        device="cuda:0", key_len_range=key_lens, out_shapes=out_shapes)
    config = {"train_micro_batch_size_per_gpu": mb, "gradient_accumulation_steps": M, "gradient_clipping": case["clip"],
              "optimizer": {"type": "Adam", "params": {"lr": 1e-5, "betas": [0.9, 0.999], "eps": 1e-8}},
              "bf16": {"enabled": dtype == torch.bfloat16}}
    engine, _, _, _ = bamboo_amd.initialize(model=model, config=config, redundancy_level=case["rc"], eager_recovery=bool(case["rc"]),
                                            activation_queue=queue, rc_stream=bool(case["rc_stream"]), install_signal_handler=False)
    for sid, sp in model.stage_params.items():
        _load(sp, seed * 7 + sid, 0.01 if kind == "decoder" else 0.02)
    if kind == "tail":
        g = torch.Generator(device="cuda:0").manual_seed(seed)
        labels = [torch.randn(mb, case["seq"], generator=g, device="cuda:0").to(dtype) for _ in range(M)]
        engine.set_dataiterator(itertools.cycle([(y, y) for y in labels]))
    queue.pipe_buffers = lambda buffers=engine: buffers.pipe_buffers
    return engine


def run(engine):
    """One batch.  Its outputs: the loss, what the stage sends to its neighbours, the redundant forwards' outputs, and the
    state after the step -- parameters, their compute copy, and both moments (the first holds the gradients)."""
    loss = engine.train_batch()
    q, sid = engine.queue, engine.stage_id
    sp = engine.module.stage_params[sid]
    return {"loss": loss, "sent": [q.sent[k] for k in sorted(q.sent)], "sent_grads": [q.sent_grads[k] for k in sorted(q.sent_grads)],
            "redundant": list(q.redundant), "master": sp.master, "compute": sp.compute, "exp_avg": sp.exp_avg,
            "exp_avg_sq": sp.exp_avg_sq}


# ------------------------------------------------------------------------------------------------ what a pass must do
def _layer_counts(case):
    """(forward flops of the stage's layers for one micro-batch, parameters, input elements, output elements)."""
    mb = case["mb"]
    if case["kind"] == "resnet":
        blocks, sides, small = _resnet_blocks(case)
        n, flops, params = case["layers"], 0, 0
        for (ci, cm, st), side in list(zip(blocks, sides))[n: 2 * n]:
            rows, out = mb * side * side, mb * ((side - 1) // st + 1) ** 2
            shortcut = st != 1 or ci != 4 * cm
            flops += 2 * rows * ci * cm + 2 * out * (9 * cm * cm + 4 * cm * cm) + (2 * out * ci * 4 * cm if shortcut else 0)
            params += ci * cm + 13 * cm * cm + 12 * cm + ((ci + 2) * 4 * cm if shortcut else 0)
        return flops, params, mb * case["side"] ** 2 * blocks[n][0], mb * small * small * 4 * case["mid"]
    h, f, s = case["hidden"], case["ffn"], case["seq"]
    rows = mb * s
    # score and context products over the pairs that the mask keeps (key lengths are uniform in [s / 4, s])
    kept = {"none": 1.0, "causal": 0.5 * (1 + 1 / s), "key_padding": 0.625}[case["mask"]]
    cross = case["kind"] == "decoder"
    flops = rows * ((16 if cross else 8) * h * h + 4 * h * f) + 4 * mb * s * s * h * (kept + (1 if cross else 0))
    params = (8 if cross else 4) * h * h + 2 * h * f + (19 if cross else 9) * h + f
    tail = case["kind"] == "tail"
    return flops * case["layers"], params * case["layers"] + (2 * h if tail else 0), rows * h, rows if tail else rows * h


def work(case):
    """Forward, twice its flops backward, and a third forward where the stage's successor is shadowed; inputs, received
    gradients and parameters read once, outputs, sent gradients and the optimizer's state written once."""
    flops, params, n_in, n_out = _layer_counts(case)
    es, M, rc = (2 if case["dtype"] == "bf16" else 4), case["M"], case["rc"]
    moved = M * es * (2 * n_in + (2 + rc) * n_out)
    state = params * (24 + (4 if es == 2 else 0)) + rc * params * es
    return {"bytes": float(moved + state), "flops": float(M * flops * (3 + rc))}


def tolerance(case):
    """bf16 storage between the kernels, several layers deep and back; where a ReLU decides on a rounded value, a decision
    may fall the other way.  fp32: sums in another order, forward and back.  (Adam turns the sign of a gradient that is
    rounding noise into a full step: single weights may be off by twice the learning rate.)"""
    if case["dtype"] == "fp32":
        return {"rel": 1e-4, "max": 2e-2}
    return {"rel": 0.03 if case["kind"] == "resnet" or case["activation"] == "relu" else 0.02, "max": 0.5}
