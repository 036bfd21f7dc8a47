"""Rules of sizes that choose between kernels, as functions of numbers alone (no GPU): where their lines lie, and that they keep to
what the kernels behind them take."""
import pytest
import torch

from infernum_amd.kernels import api as K


# tokens from which routed experts take the grouped product: 112 pairs an expert, 56 for wide experts that fill the chip (both sides
# of either condition) and without a gate; never where that product does not take the sizes
@pytest.mark.parametrize("E,top,W,ff,gated,tokens", [
    (32, 4, 2048, 1408, True, 896), (20, 2, 4096, 2432, True, 560), (8, 2, 4096, 4800, True, 224), (8, 2, 4096, 14336, True, 224),
    (4, 2, 4096, 4800, True, 224), (5, 1, 4096, 4800, True, 560), (6, 1, 4096, 4800, True, 336), (8, 2, 2048, 2752, True, 448),
    (8, 2, 3072, 2880, True, 448), (10, 2, 3072, 2944, True, 280), (8, 3, 2048, 2752, False, 150), (8, 2, 4096, 4800, False, 224),
    (8, 2, 2040, 2752, True, 0), (8, 2, 2048, 2744, False, 0)])
def test_tokens_from_which_experts_take_the_grouped_product(E, top, W, ff, gated, tokens):
    assert K.moe_grouped_from_tokens(E, top, W, ff, torch.bfloat16, gated) == tokens
    assert K.moe_grouped_from_tokens(E, top, W, ff, torch.float32, gated) == 0
    if tokens:
        assert K.moe_grouped_rows(tokens, E, top, W, ff, torch.bfloat16, gated)
        assert not K.moe_grouped_rows(tokens - 1, E, top, W, ff, torch.bfloat16, gated)


# parts of the keys in decode attention on 256 compute units: whole up to 256 keys and where the requests fill the chip; heads up to 64: a
# workgroup a unit up to 8,192 keys where that is four parts or more, two from there on, 32 parts at the most; up to 128: three quarters of
# the units only in place of all of them; above: a part for four tiles
@pytest.mark.parametrize("batch,nkv,head,keys,parts", [
    (1, 8, 64, 256, 1), (64, 8, 64, 4000, 1), (20, 8, 128, 4000, 1),
    (1, 8, 64, 8192, 32), (1, 8, 64, 32768, 32), (2, 8, 64, 4096, 16), (2, 8, 64, 32768, 32), (4, 8, 64, 1024, 8), (8, 8, 64, 528, 4),
    (8, 8, 64, 32768, 8), (9, 8, 64, 1024, 7), (12, 8, 64, 528, 5), (1, 8, 64, 300, 3),
    (4, 8, 128, 8192, 6), (3, 8, 128, 8192, 10), (3, 4, 128, 32768, 21), (2, 8, 128, 4096, 12), (1, 8, 128, 4096, 24), (8, 8, 128, 528, 4),
    (16, 2, 96, 8192, 8), (1, 1, 256, 1024, 16), (1, 1, 256, 16384, 64), (32, 1, 256, 2048, 8)])
def test_parts_of_the_keys_in_decode_attention(monkeypatch, batch, nkv, head, keys, parts):
    monkeypatch.setattr(K, "compute_units", lambda device=None: 256)
    assert K.decode_splits(batch, 4 * nkv, nkv, keys, None, head) == parts


@pytest.mark.parametrize("cap", [-30.0, float("nan")])
def test_a_softcap_that_is_not_positive_is_no_empty_finish(cap):
    """... so that the launch or the function that applies it refuses it, as before it was applied on the way to memory."""
    from infernum_amd.parts.linear import Finish
    assert Finish(cap=cap) and not Finish() and Finish(cap=2.0) and Finish(scale=0.5)
    with pytest.raises(K.KernelError):
        Finish(cap=cap).apply(torch.zeros(2, 8))
