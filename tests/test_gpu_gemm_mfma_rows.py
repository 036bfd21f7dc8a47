"""The split product and the one with the activation on either side of 64 rows, from where on their tiles are larger: the same bits."""
import math

import pytest
import torch

pytestmark = pytest.mark.gpu
DEV = "cuda"


def _rand(*shape, scale=1.0, seed=0):
    g = torch.Generator(device=DEV).manual_seed(seed)
    return (torch.randn(*shape, device=DEV, generator=g) * scale).to(torch.bfloat16)


# columns of one tile, of one and some; one step of K, fewer steps than stages, more; parts of unequal length
@pytest.mark.parametrize("N,K_,S", [(96, 64, 1), (130, 128, 2), (770, 704, 3), (256, 1024, 1)])
def test_up_to_64_rows_as_with_more(N, K_, S):
    from infernum_amd.kernels import api
    a, w = _rand(65, K_, seed=1), _rand(N, K_, scale=0.1, seed=2)
    want = a.double() @ w.double().t()
    of_65 = api.gemm_mfma_split(a, w, S).parts
    # fp32 sums of K_ products, each addition within 2^-24 of the running sum, of the order of 0.1 sqrt(K)
    assert bool(((of_65.double().sum(0) - want).abs() <= 2e-5 * math.sqrt(K_) * 0.1).all())
    act = api.gemm_mfma_swiglu(a, w)
    tiled = api.tile_weight(w, "swiglu") if api.gemm_skinny_splits(N, K_) == 1 else None
    for M in (64, 63, 33, 32, 1):
        parts = torch.full((S + 1, M, N), 7.0, device=DEV)
        assert torch.equal(api.gemm_mfma_split(a[:M].contiguous(), w, S, parts[:S]).parts, of_65[:, :M]), M
        assert bool((parts[S] == 7.0).all())                             # nothing behind the last part
        assert torch.equal(api.gemm_mfma_swiglu(a[:M].contiguous(), w), act[:M]), M
        if tiled is not None:
            assert torch.equal(api.gemm_mfma_swiglu(a[:M].contiguous(), w, tiled=tiled), act[:M]), M


# as many tiles of 64 x 64 as there are compute units and one more (tiles of 64 x 128); columns that fill no tile; fewer steps of K than
# stages, and more
@pytest.mark.parametrize("N,K_,S", [(16380, 128, 1), (16386, 128, 1), (2040, 3200, 8), (2060, 640, 8)])
def test_up_to_64_rows_by_how_many_tiles_there_are(N, K_, S):
    from infernum_amd.kernels import api
    a, w = _rand(129, K_, seed=5), _rand(N, K_, scale=0.1, seed=6)
    of_129 = api.gemm_mfma_split(a, w, S).parts
    want = a.double() @ w.double().t()
    assert bool(((of_129.double().sum(0) - want).abs() <= 2e-5 * math.sqrt(K_) * 0.1).all())
    for M in (64, 33, 17, 1):
        parts = torch.full((S + 1, M, N), 7.0, device=DEV)
        assert torch.equal(api.gemm_mfma_split(a[:M].contiguous(), w, S, parts[:S]).parts, of_129[:, :M]), M
        assert bool((parts[S] == 7.0).all())


def test_the_head_of_many_columns_from_17_rows_on():
    """An fp32 result as wide as fills the chip by the tiled kernel from 17 rows on, in the plan and in what linear gives; each row as
    near to 64 bits as by the weight-streaming kernel, and the same whatever stands beside it."""
    import importlib
    from infernum_amd.kernels import api
    L = importlib.import_module("infernum_amd.parts.linear")
    N, K_ = L.FP32_TILED_WIDE, 1088
    kinds = [L.route_of(L.plan(n, K_, torch.bfloat16, torch.float32, None, False), m).kind for n, m in ((N, 16), (N, 17), (N - 1, 17))]
    assert kinds == ["skinny", "mfma_f32", "skinny"]
    x, w = _rand(33, K_, seed=3), _rand(N, K_, scale=0.1, seed=4)
    want = x.double() @ w.double().t()
    y = L.linear(x, w, out_dtype=torch.float32)
    few = api.gemm_skinny(x, w, out_dtype=torch.float32)
    assert y.dtype == torch.float32 and bool(((y.double() - want).abs() <= 2e-5 * math.sqrt(K_) * 0.1).all())
    a, b = ((t.double() - want).pow(2).mean().sqrt().item() for t in (y, few))
    assert a <= 1.25 * b, (a, b)
    assert torch.equal(L.linear(x[:17].contiguous(), w, out_dtype=torch.float32), y[:17])


# as many tiles of 32 x 64 as the rule takes (a row more of tiles: tiles of 128 x 128), rows and columns that fill no tile, fewer steps of
# K than stages
@pytest.mark.parametrize("M,N,K_,S", [(65, 5, 64, 1), (1248, 770, 448, 1), (8192, 120, 192, 1), (607, 770, 320, 2)])
def test_few_columns_as_with_more_rows(M, N, K_, S):
    from infernum_amd.kernels import api
    tiles = -(-M // 32) * -(-N // 64) * S
    more = M + 32 * (-(-(513 - tiles) // (-(-N // 64) * S)))
    assert tiles <= 512 < -(-more // 32) * -(-N // 64) * S
    a, w = _rand(more, K_, seed=7), _rand(N, K_, scale=0.1, seed=8)
    want = a[:M].double() @ w.double().t()
    parts = torch.full((S + 1, M, N), 7.0, device=DEV)
    got = api.gemm_mfma_split(a[:M].contiguous(), w, S, parts[:S]).parts
    assert bool(((got.double().sum(0) - want).abs() <= 2e-5 * math.sqrt(K_) * 0.1).all()) and bool((parts[S] == 7.0).all())
    assert torch.equal(api.gemm_mfma_split(a, w, S).parts[:, :M], got)
