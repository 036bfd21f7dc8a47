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
