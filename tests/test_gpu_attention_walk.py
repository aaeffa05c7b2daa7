"""Attention backward whose waves look one sub-tile ahead: lengths around the edges of sub-tiles (32), tiles (64) and blocks, walks of one,
two and three tiles (the ring's stages), padding that ends inside a sub-tile, queries and keys past the end in the last block;
against fp64, twice the same bits, without and with dropout."""
import pytest
import torch

from tests import test_gpu_dropout as drop
from tests import test_gpu_kernels as plain

pytestmark = pytest.mark.gpu

SHAPES = [(1, 2, 31, 64), (2, 1, 32, 64), (1, 3, 33, 64), (1, 2, 63, 32), (2, 2, 65, 32), (1, 2, 96, 128), (1, 1, 97, 64), (3, 2, 129, 64),
          (1, 4, 191, 32), (2, 6, 385, 32), (1, 150, 70, 64), (1, 24, 1025, 64), (2, 260, 161, 64), (1, 600, 129, 64)]   # the last two beyond a round


@pytest.mark.parametrize("mask", ["none", "causal", "key_padding"])
@pytest.mark.parametrize("b,a,s,d", SHAPES)
def test_walk(hiplib, mask, b, a, s, d):
    plain.test_fused_attention_fwd_bwd(hiplib, mask, b, a, s, d)


@pytest.mark.parametrize("mask", ["none", "causal", "key_padding"])
@pytest.mark.parametrize("b,a,s,d", [t for t in SHAPES if t[0] <= 2 and 63 <= t[2] and t[1] < 100])   # (its key lengths: 37 short of all)
def test_walk_with_dropout(hiplib, mask, b, a, s, d):
    drop.test_fused_attention_dropout_fwd_bwd(hiplib, mask, b, a, s, d)


@pytest.mark.parametrize("mask", ["none", "causal", "key_padding"])
@pytest.mark.parametrize("b,a,s,d", [(1, 1, 1, 64), (2, 2, 33, 64), (2, 4, 67, 32), (1, 2, 128, 64), (1, 2, 161, 128), (1, 2, 515, 64), (2, 6, 200, 32),
                                     (2, 130, 200, 64), (2, 40, 461, 128), (1, 40, 530, 64),
                                     # walks shared by groups: 2x4 in one launch and in two, 2x2, 4x2; pairs of heads 2x2; 128-wide 4x2
                                     (1, 2, 600, 64), (1, 2, 2100, 64), (2, 8, 520, 64), (1, 22, 450, 64), (1, 9, 1210, 64), (1, 11, 1537, 64),
                                     (2, 16, 600, 32), (1, 2, 500, 128), (1, 30, 500, 128)])
def test_kept_decisions(hiplib, mask, b, a, s, d):
    """The backward that reads the forward's decisions against the one that makes them again: the same bits; the forward does not
    change by keeping them."""
    g = torch.Generator(device="cuda").manual_seed(5)
    qkv, d_out = (torch.randn(b * s, w, generator=g, device="cuda").bfloat16() for w in (3 * a * d, a * d))
    lens = torch.tensor([max(1, s - 37), s][:b], dtype=torch.int32, device="cuda") if mask == "key_padding" else None
    keep = torch.full((hiplib.attention_keep_words(b, a, s),), -1, dtype=torch.int32, device="cuda")
    args, drop_key = (b, a, s, hiplib.MASK_CODES[mask], lens), (0.3, (77, 99))
    result = []
    for kept in (None, keep):
        out, lse, delta = torch.empty_like(d_out), torch.empty(b, a, s, device="cuda"), torch.empty(b, a, s, device="cuda")
        d_qkv = torch.full_like(qkv, float("nan"))
        hiplib.attention_fwd(qkv, out, lse, *args, dropout=drop_key, keep=kept)
        hiplib.attention_bwd(qkv, out, d_out, lse, delta, d_qkv, *args, dropout=drop_key, keep=kept)
        result.append((out, lse, d_qkv))
    assert all(torch.equal(x, y) for x, y in zip(*result))
    assert torch.isfinite(result[0][2]).all()
    with pytest.raises(hiplib.HipKernelError, match="keep"):
        hiplib.attention_fwd(qkv, out, lse, *args, dropout=drop_key, keep=keep[1:])
