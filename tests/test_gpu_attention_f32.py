"""The fp32 attention kernels that keep the probabilities, where they can go wrong: sequences around the 32-wide tiles and the
64-wide steps of the row pass, one head width per instantiation, masks with empty and one-key rows, dropout; against fp64 autograd
and against the batched products that run the other shapes."""
import math

import pytest
import torch

from bamboo_amd import TransformerLayer, hip

DEV = "cuda:0"


def test_shapes_the_kernels_take():
    """Decided on the host: fp32, three head widths, whole 16-byte vectors of probabilities, rows that fit the strip in LDS."""
    ok = lambda *a: hip.attention_probs_supported(*a)
    f32 = torch.float32
    assert ok(f32, 1, 1, 4, 32) and ok(f32, 2, 3, 1024, 64) and ok(f32, 1, 1, 256, 128)
    assert not ok(torch.bfloat16, 1, 1, 64, 64) and not ok(f32, 1, 1, 64, 96) and not ok(f32, 1, 1, 66, 64)
    assert not ok(f32, 1, 1, 1028, 64) and not ok(f32, 1, 4096, 64, 64)
    assert not ok(f32, 1, 4, 512, 128) and ok(f32, 1, 6, 512, 128)
    L = hip.lib()
    assert L.bb_attention_probs_fwd(0, 0, 1, 1, 66, 64, 16, 16, 16, 192, 16, 64, 16, None, 0.0, 0, 0, None) == -1
    assert b"multiple of 4" in L.bb_last_error()
    assert L.bb_attention_probs_fwd(0, 0, 1, 1, 64, 64, 16, 16, 20, 192, 16, 64, 16, None, 0.0, 0, 0, None) == -1
    assert b"aligned" in L.bb_last_error()


def _run(layer, ctx, qkv, d_ctx):
    b, a, s = ctx.batch, layer.heads, ctx.seq
    ctx.ensure_scratch(layer.scratch_specs(ctx))
    for t in ctx.scratch.values():
        t.fill_(float("nan"))
    st = {"qkv": qkv, "ctx": torch.full_like(d_ctx, float("nan")), "prob": torch.full((b, a, s, s), float("nan"), device=DEV)}
    d_qkv = torch.full_like(qkv, float("nan"))
    layer._attention_fwd(st, ctx)
    layer._attention_bwd(d_ctx, d_qkv, st, ctx)
    torch.cuda.synchronize()
    return st["prob"], st["ctx"], d_qkv


@pytest.mark.gpu
@pytest.mark.parametrize("mask", ["none", "causal", "key_padding"])
@pytest.mark.parametrize("b,a,s,d,p", [(1, 1, 4, 64, 0.0), (3, 3, 36, 32, 0.1), (2, 2, 64, 64, 0.0), (3, 5, 100, 128, 0.1), (3, 3, 132, 64, 0.1),
                                       (3, 2, 288, 32, 0.0), (4, 6, 516, 128, 0.0), (3, 1, 1024, 64, 0.1)])
def test_kept_probabilities(hiplib, mask, b, a, s, d, p):
    from bamboo_amd.layers import StageContext
    h = a * d
    g = torch.Generator(device=DEV).manual_seed(5)
    qkv = torch.randn(b * s, 3 * h, generator=g, device=DEV) * 0.7
    d_ctx = torch.randn(b * s, h, generator=g, device=DEV)
    # the first of several samples has no key at all, the next one
    lens = torch.tensor([0, 1, s, s][:b] if b > 1 else [s - 1], dtype=torch.int32, device=DEV) if mask == "key_padding" else None
    got = []
    for kernels in (True, False):
        layer = TransformerLayer(h, a, 4 * h, mask=mask, dropout=p, activation="gelu_tanh")
        layer.layer_idx = 3
        ctx = StageContext(b, s, torch.float32, torch.device(DEV))
        ctx.key_len, ctx.dropout_base = lens, (11, 2, 1)
        assert layer.kept_probs_kernels(ctx)
        if not kernels:
            layer.kept_probs_kernels = lambda ctx: False
        got.append(_run(layer, ctx, qkv, d_ctx))
    x = qkv.double().cpu().requires_grad_(True)
    q, k, v = [x[:, i * h:(i + 1) * h].view(b, s, a, d).transpose(1, 2) for i in range(3)]
    scores = q @ k.transpose(-2, -1) / math.sqrt(d)
    if mask == "causal":
        scores = scores.masked_fill(~torch.tril(torch.ones(s, s, dtype=torch.bool)), -1e9)
    elif mask == "key_padding":
        scores = scores.masked_fill(~(torch.arange(s).view(1, 1, 1, s) < lens.cpu().view(b, 1, 1, 1)), -1e9)
    prob = torch.softmax(scores, -1)
    kept = prob
    if p:
        ones = torch.ones(b, a, s, s, device=DEV)
        keep = torch.empty_like(ones)
        hip.dropout_apply(ones, keep, p, layer._drop(ctx, 0)[1])
        kept = prob * keep.double().cpu()
    out = (kept @ v).transpose(1, 2).reshape(b * s, h)
    out.backward(d_ctx.double().cpu())
    want = [prob.detach(), out.detach()] + [x.grad[:, i * h:(i + 1) * h] for i in range(3)]
    # roundings of chains of `d` and of `s` fp32 additions add up like a random walk; a few more for the row operations
    tol = 2.0 ** -24 * (math.sqrt(d) + math.sqrt(s) + 8)
    floor = 1e-3 * float(x.grad.norm())     # a causal row with one key has no gradient but rounding
    # without a key all probabilities are equal; what they then pass on to the scores autograd's masked_fill would stop, the
    # softmax backward of the products does not: such a sample's gradients are compared between the two ways only
    seen = slice(1 if mask == "key_padding" and b > 1 else 0, None)
    pick = lambda t, part: t.reshape(b, -1)[part].double().cpu()
    parts = [[pr, c] + [dq[:, i * h:(i + 1) * h] for i in range(3)] for pr, c, dq in got]
    for which, ts in zip(("kernels", "products"), parts):
        for name, t, w in zip(("prob", "ctx", "dq", "dk", "dv"), ts, want):
            part = seen if name[0] == "d" else slice(None)
            err = float((pick(t, part) - pick(w, part)).norm()) / max(float(pick(w, part).norm()), floor if name[0] == "d" else 0.0)
            assert err < tol, (which, name, err, tol)
    for name, t, w in zip(("prob", "ctx", "dq", "dk", "dv"), *parts):
        err = float((t - w).double().norm()) / max(float(w.double().norm()), floor if name[0] == "d" else 0.0)
        assert err < 2 * tol, (name, err, tol)
    assert torch.equal(got[0][0] == 0, got[1][0] == 0)      # the masked probabilities, exactly


@pytest.mark.gpu
@pytest.mark.parametrize("mask", ["none", "causal", "key_padding"])
@pytest.mark.parametrize("b,a,s,d", [(1, 1, 4, 32), (2, 2, 36, 64), (1, 3, 100, 128), (2, 1, 132, 64)])
def test_nothing_past_the_end_is_taken_in(hiplib, mask, b, a, s, d):
    """A ragged sequence is read in whole tiles: what lies behind the operands, of a sample or of all of them, reads as zero.  With
    NaN there, and without: the same bits."""
    h, n = a * d, b * s
    g = torch.Generator(device=DEV).manual_seed(s)
    rand = lambda *shape: torch.randn(*shape, generator=g, device=DEV)
    qkv, d_ctx = rand(n, 3 * h), rand(n, h)
    lens = torch.tensor([s - 1, s][:b], dtype=torch.int32, device=DEV) if mask == "key_padding" else None
    runs = []
    for behind in (0.0, float("nan")):
        pad = lambda t: torch.cat([t.reshape(-1), torch.full((64 * t.shape[-1],), behind, device=DEV)])[: t.numel()].view(t.shape)
        new = lambda *shape: pad(torch.full(shape, float("nan"), device=DEV))
        q, dc, out, prob, d_score, d_qkv = pad(qkv), pad(d_ctx), new(n, h), new(b, a, s, s), new(b, a, s, s), new(n, 3 * h)
        hip.attention_probs_fwd(q, out, prob, b, a, s, hip.MASK_CODES[mask], lens)
        hip.attention_probs_bwd(q, dc, prob, d_score, d_qkv, b, a, s, hip.MASK_CODES[mask], lens)
        runs.append((out, prob, d_qkv))
    for x, y in zip(*runs):
        assert bool(torch.isfinite(x).all()) and torch.equal(x, y)
