"""Dropout inside the fused attention at sequence lengths whose rows start inside a hash pair, and at short and ragged ones (the shorter batch entry keeps seq - 37 keys)."""
import pytest

from tests import test_gpu_dropout as even

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("mask", ["none", "causal", "key_padding"])
@pytest.mark.parametrize("batch,heads,seq,d", [(1, 3, 175, 64), (2, 2, 39, 64), (2, 4, 77, 32), (1, 1, 129, 128), (2, 1, 38, 64), (1, 2, 98, 32)])
def test_odd_and_ragged_sequences(hiplib, mask, batch, heads, seq, d):
    even.test_fused_attention_dropout_fwd_bwd(hiplib, mask, batch, heads, seq, d)
