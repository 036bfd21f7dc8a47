"""The products of a prompt's rows in quadrants (csrc/gemm_tiles.hip) against plain products in 64 bits, at the edges of their tiles."""
import importlib
import math

import pytest
import torch

pytestmark = pytest.mark.gpu
DEV = "cuda"


def K():
    from infernum_amd.kernels import api
    return api


def _rand(*shape, scale=1.0, seed=0):
    g = torch.Generator(device=DEV).manual_seed(seed)
    return (torch.randn(*shape, device=DEV, generator=g) * scale).to(torch.bfloat16)


TILES = K().GEMM_TILES


@pytest.mark.parametrize("tile", TILES)
@pytest.mark.parametrize("M,N,K_", [(1, 8, 64), (257, 516, 128), (300, 1003, 192), (515, 771, 448), (129, 250, 576)])
def test_whole_products_at_sizes_that_fill_no_tile(tile, M, N, K_):
    """One row and one step of K; an odd and an even number of steps; edges in M and N; columns off 16 bytes."""
    api = K()
    a, w = _rand(M, K_, seed=1), _rand(N, K_, scale=0.1, seed=2)
    want = a.double() @ w.double().t()
    out = torch.full((M + 1, N), float("nan"), dtype=torch.bfloat16, device=DEV)
    api.gemm_tiles(a, w, out[:M], tile=tile)
    # fp32 sums of K_ products (each addition within 2^-24 of the running sum, of the order of 0.1 sqrt(K)), one rounding to bf16
    bound = 2e-5 * math.sqrt(K_) * 0.1 + 2.0 ** -8 * want.abs()
    assert bool(((out[:M].double() - want).abs() <= bound).all())
    assert bool(out[M].isnan().all())                                   # nothing behind the last row
    # a row's result depends neither on the rows beside it nor on the tile: the sums run over K in its order
    assert torch.equal(api.gemm_tiles(a[M - 1:M].clone(), w, tile=tile)[0], out[M - 1])
    assert torch.equal(api.gemm_tiles(a, w), out[:M])
    assert torch.equal(api.gemm_mfma(a, w, tile="128x128"), out[:M])


@pytest.mark.parametrize("tile", [t for t in TILES if t[1] not in (224, 160)])
@pytest.mark.parametrize("M,N,K_", [(1, 16, 64), (300, 1004, 192), (515, 770, 448)])
def test_products_with_the_activation(tile, M, N, K_):
    api = K()
    a, w = _rand(M, K_, seed=3), _rand(N, K_, scale=0.2, seed=4)
    g, u = (a.double() @ w.double().t()).split(N // 2, dim=1)
    want = g * torch.sigmoid(g) * u
    out = api.gemm_tiles(a, w, swiglu=True, tile=tile)
    # the sums' errors e through silu' <= 1.1 and the other factor, the activation's few 2^-24, one rounding to bf16
    e = 2e-5 * math.sqrt(K_) * 0.2
    bound = e * (1.1 * u.abs() + g.abs()) + 1e-6 * want.abs() + 2.0 ** -8 * want.abs() + 1e-6
    assert bool(((out.double() - want).abs() <= bound).all())
    assert torch.equal(api.gemm_tiles(a[M - 1:M].clone(), w, swiglu=True)[0], out[M - 1])


def test_the_activation_at_its_ends():
    """Gates that saturate to either side give what silu(g) u gives in 64 bits (0 and u g)."""
    api = K()
    gates = torch.tensor([-3e4, -200.0, -90.0, -20.0, 0.0, 20.0, 200.0, 3e4], device=DEV)
    a = torch.zeros(8, 64, dtype=torch.bfloat16, device=DEV)
    a[:, 0], a[:, 1] = gates.to(torch.bfloat16), 1.0
    w = torch.zeros(32, 64, dtype=torch.bfloat16, device=DEV)
    w[:16, 0], w[16:, 1] = 1.0, 2.0
    out = api.gemm_tiles(a, w, swiglu=True)
    g = a[:, :1].double()
    want = (g * torch.sigmoid(g) * 2.0).expand(8, 16)
    assert bool(((out.double() - want).abs() <= 2.0 ** -8 * want.abs() + 1e-7).all())


def test_one_product_is_picked_out():
    """Single entries at the ends of rows, columns and K: a wrong place in LDS, half-tile or step would move or lose one."""
    api = K()
    M, N, K_ = 515, 771, 448
    a = torch.zeros(M, K_, dtype=torch.bfloat16, device=DEV)
    w = torch.zeros(N, K_, dtype=torch.bfloat16, device=DEV)
    for i, (m, n, k) in enumerate([(0, 0, 0), (M - 1, N - 1, K_ - 1), (256, 255, 64), (129, 513, 71), (300, 2, 447), (63, 127, 320)]):
        a[m, k] = 1 + i
        w[n, k] = 2
    want = a.float() @ w.float().t()
    for tile in TILES:
        assert torch.equal(api.gemm_tiles(a, w, tile=tile).float(), want), tile


def test_what_it_refuses():
    api = K()
    a, w = _rand(70, 96), _rand(32, 96)
    with pytest.raises(api.KernelError):
        api.gemm_tiles(a, w)                                                            # K % 64
    a, w = _rand(70, 128), _rand(33, 128)
    with pytest.raises(api.KernelError):
        api.gemm_tiles(a, w, swiglu=True)                                               # halves of an odd number
    with pytest.raises(api.KernelError):
        api.gemm_tiles(a, w, tile=(64, 64))
    off = torch.zeros(33 * 128 + 4, dtype=torch.bfloat16, device=DEV)[4:].view(33, 128)
    with pytest.raises(api.KernelError):
        api.gemm_tiles(a, off)                                                          # off 16 bytes


# columns in two launches of a tile each, the last of either in part: the same bits as one tile for all, and nothing stored twice or beyond
@pytest.mark.parametrize("M,N,K_,swiglu", [(1125, 16392, 1024, False), (1146, 17122, 2048, True), (1121, 17634, 2048, True), (1009, 16762, 3072, False)])
def test_columns_in_two_launches_leave_the_bits_of_one(M, N, K_, swiglu):
    api = K()
    a, w = _rand(M, K_, seed=21), _rand(N, K_, scale=0.1, seed=22)
    cols = N // 2 if swiglu else N
    assert 0 < api._core().ia_gemm_tiles_split(M, N, K_, int(swiglu)) < cols
    out = torch.full((M + 1, cols), 7.0, dtype=torch.bfloat16, device=DEV)
    api.gemm_tiles(a, w, out[:M], swiglu=swiglu)
    assert torch.equal(out[:M], api.gemm_tiles(a, w, swiglu=swiglu, tile=(128, 128)))
    assert bool((out[M:] == 7.0).all())


@pytest.mark.parametrize("off", [False, True])
@pytest.mark.parametrize("M,N,K_", [(300, 512, 256), (2304, 2048, 2048), (2304, 2304, 4096)])
def test_many_rows_take_it_where_it_is_the_faster(M, N, K_, off):
    """The many-row route, plain and with the activation, for weights on 16 bytes and off them (the library's then)."""
    L = importlib.import_module("infernum_amd.parts.linear")   # the package exports the function under this name
    api = K()
    x = _rand(M, K_, seed=5)
    raw = torch.empty(N * K_ + 8, dtype=torch.bfloat16, device=DEV)
    w = raw[4:4 + N * K_].view(N, K_) if off else raw[:N * K_].view(N, K_)
    w.copy_(_rand(N, K_, scale=0.1, seed=6))
    for epilogue in (None, "swiglu"):
        assert L.route_of(L.plan(N, K_, torch.bfloat16, torch.bfloat16, epilogue, False), M).kind == "library"
        y = L.linear(x, w, epilogue=epilogue)
        want = x.double() @ w.double().t()
        if epilogue:
            g, u = want.split(N // 2, dim=1)
            want = g * torch.sigmoid(g) * u
        # with the activation behind the library's product gate, up and result are rounded to bf16
        assert float((y.double() - want).norm() / want.norm()) < (6e-3 if epilogue else 3e-3)
        if not off and (epilogue or api.gemm_tiles_pays(M, N, K_)):
            assert torch.equal(y, api.gemm_tiles(x, w.clone(), swiglu=bool(epilogue)))


@pytest.mark.parametrize("M,N,K_", [(2048, 4096, 14336), (8192, 4096, 14336), (7650, 4096, 14336), (512, 4096, 14336), (1500, 6144, 4096),
                                   (300, 4096, 4096), (5700, 2048, 2048), (2300, 2048, 8192), (3000, 2048, 2048), (2048, 4096, 1984),
                                   (2048, 4096, 4100), (70000, 4096, 32768), (4600, 10240, 8192), (7650, 4096, 10240)])
def test_where_whole_products_take_it(M, N, K_):
    """The rule of sizes against itself written plainly."""
    api = K()
    large, small = math.ceil(M / 256) * math.ceil(N / 256), math.ceil(M / 128) * math.ceil(N / 128)
    empty = math.ceil(large / 256) * 256 / large
    want = (K_ % 64 == 0 and max(M, N) * K_ * 2 < 2 ** 32 - 3072 and small >= 200 and K_ >= 2048 and (K_ >= 4096 or large <= 140)
            and empty >= (1.06 if K_ >= 10240 and large > 256 else 1.2))
    assert api.gemm_tiles_pays(M, N, K_) == want


# rows of the groups (and how often these repeat), columns, K: a tile's last row and one more, one row, none; columns that fill no tile, of
# two starts of the walk, off 16 bytes
@pytest.mark.parametrize("counts,times,N,K_", [((96, 97, 0, 1, 95, 192), 1, 200, 64), ((3,), 1, 130, 320), ((96, 97, 0, 1, 95, 64), 6, 1032, 192),
                                               ((160, 161, 0, 1, 159, 300), 6, 1032, 320), ((192, 193, 0, 1, 191, 500), 6, 1032, 448)])
def test_rows_in_groups_at_the_edges_of_each_tile(counts, times, N, K_):
    api = K()
    counts = list(counts) * times
    rows, G = sum(counts) + 2, len(counts)
    x, w = _rand(rows, K_, seed=5), _rand(G, N, K_, scale=0.1, seed=6)
    at = torch.tensor([0] + counts, device=DEV).cumsum(0).int()
    out = torch.full((rows, N), 7.0, dtype=torch.bfloat16, device=DEV)
    api.gemm_mfma_grouped(x, w, at, out)
    lo = 0
    for g, n in enumerate(counts):
        want = x[lo:lo + n].double() @ w[g].double().t()
        # as for whole products above
        assert bool(((out[lo:lo + n].double() - want).abs() <= 2e-5 * math.sqrt(K_) * 0.1 + 2.0 ** -8 * want.abs()).all()), g
        if n:                                                            # the first 512 columns begin their walk over K at 0
            assert torch.equal(out[lo:lo + n, :512], api.gemm_tiles(x[lo:lo + n].clone(), w[g])[:, :512]), g
        lo += n
    assert bool((out[lo:] == 7.0).all())


# a matrix whose tiles fill half the compute units (few rows to the library, with more rows here), one column tile more, one of short K
@pytest.mark.parametrize("N,K_,first", [(16384, 2048, 129), (16512, 2048, 1), (16384, 1024, 1), (10752, 5120, 257), (2816, 1536, 257)])
def test_where_products_with_the_activation_take_it(N, K_, first):
    """The rule against itself written plainly, and what the route returns on both sides of its line."""
    L = importlib.import_module("infernum_amd.parts.linear")
    api = K()
    assert L.glu_tiles_from(N, K_) == first
    for M in (*range(1, 700, 7), 128, 129, 256, 257, 3000):
        tiles = math.ceil(M / 128) * math.ceil(N / 128)
        assert (M >= first) == (K_ * (256 - tiles) < 2 ** 18 or (K_ <= 2048 and M > 128 and tiles > 64)), M
    w = _rand(N, K_, scale=0.05, seed=8)
    routes = L.plan(N, K_, torch.bfloat16, torch.bfloat16, "swiglu", False)
    for M in (65, 96, 129, 257):
        if L.route_of(routes, M).kind != "library":
            continue
        x = _rand(M, K_, seed=M)
        y = L.linear(x, w, epilogue="swiglu")
        if M >= first:
            want = api.gemm_tiles(x, w, swiglu=True)
        else:
            want = api.swiglu(api.gemm_library(x, w), torch.empty((M, N // 2), dtype=torch.bfloat16, device=DEV))
        assert torch.equal(y, want), M


def test_the_activation_where_its_sums_are_infinite_or_its_sigmoid_is_tiny():
    """Sums of +-inf and NaN give what silu(g) u gives in fp32; a sigmoid below the smallest normal number is not lost: to -88.5 the product
    is that of 64 bits, and further down, where exp(-g) leaves fp32, it is that or 0."""
    api = K()
    inf = float("inf")
    gates = torch.tensor([inf, -inf, float("nan"), -86.0, -87.0, -87.5, -88.0, -88.5, -89.0, -90.0, -95.0, -104.0, -3e38], device=DEV)
    n = gates.numel()
    a = torch.zeros(n, 64, dtype=torch.bfloat16, device=DEV)
    a[:, 0], a[:, 1] = gates.to(torch.bfloat16), 1.0
    w = torch.zeros(32, 64, dtype=torch.bfloat16, device=DEV)
    w[:16, 0], w[16:, 1] = 1.0, 2.0
    w[16:, 0] = 0.0
    out = api.gemm_tiles(a, w, swiglu=True).double()
    g = a[:, 0].double()
    g[:3] = gates[:3].double()
    want = (g * torch.sigmoid(g) * 2.0)[:, None].expand(n, 16)
    # an infinite or NaN value times the weights' zeros makes up NaN as well: the gate's own sum stays what it is only in the products' first
    # factor, so that row 0 to 2 are NaN whatever the activation does; the rest is finite
    assert bool(out[:3].isnan().all()) and bool(out[3:].isfinite().all())
    assert bool(((out[3:8] - want[3:8]).abs() <= 2.0 ** -7 * want[3:8].abs()).all())
    assert bool(((out[8:] - want[8:]).abs() <= 2.0 ** -7 * want[8:].abs()).logical_or(out[8:] == 0).all())
    # sums that are infinite by themselves: 2 x 3e38
    big = torch.full((4, 64), 0.0, dtype=torch.bfloat16, device=DEV)
    big[:, 0] = big[:, 1] = torch.tensor([3e38, -3e38, 3e38, -3e38], device=DEV).to(torch.bfloat16)
    big[:, 2] = torch.tensor([1.0, 1.0, -1.0, 0.0], device=DEV).to(torch.bfloat16)
    w = torch.zeros(32, 64, dtype=torch.bfloat16, device=DEV)
    w[:16, :2], w[16:, 2] = 1.0, 2.0
    out = api.gemm_tiles(big, w, swiglu=True).float()
    g, u = (big.float() @ w.float().t()).split(16, dim=1)
    assert bool(g.isinf().all()) and torch.equal(torch.nan_to_num(out, nan=7.0), torch.nan_to_num(torch.nn.functional.silu(g) * u, nan=7.0))


# every tile that the choice can fall on: the mean rows of so many groups that lead to it
@pytest.mark.parametrize("tile,groups,mean,N,K_", [((96, 128), 12, 50, 200, 192), ((128, 128), 32, 104, 1034, 64), ((160, 128), 16, 141, 2056, 64),
                                                   ((192, 128), 16, 176, 2056, 64), ((128, 256), 8, 623, 1034, 2752),
                                                   ((192, 256), 8, 827, 1290, 2752), ((256, 256), 8, 884, 1546, 1024)])
def test_each_tile_of_rows_in_groups(tile, groups, mean, N, K_):
    """Groups of a tile's rows, one more and one less, of one row and of none, the others such that the mean is kept."""
    api = K()
    bm = tile[0]
    assert api._core().ia_gemm_tiles_grouped_tile(groups, mean, N, K_) == bm * 1024 + tile[1]
    counts = [bm, bm + 1, 0, 1, bm - 1, 2 * bm]
    left = mean * groups - sum(counts)
    counts += [left // (groups - 6)] * (groups - 7)
    counts.append(mean * groups - sum(counts))
    assert min(counts) >= 0 and sum(counts) // groups == mean
    x, w = _rand(sum(counts), K_, seed=5), _rand(groups, N, K_, scale=0.1, seed=6)
    at = torch.tensor([0] + counts, device=DEV).cumsum(0).int()
    out = torch.full((sum(counts), N), 7.0, dtype=torch.bfloat16, device=DEV)
    api.gemm_mfma_grouped(x, w, at, out)
    lo = 0
    for g, n in enumerate(counts):
        want = x[lo:lo + n].double() @ w[g].double().t()
        # as for whole products above
        assert bool(((out[lo:lo + n].double() - want).abs() <= 2e-5 * math.sqrt(K_) * 0.1 + 2.0 ** -8 * want.abs()).all()), g
        if n and g < 8:                                                 # the first 512 columns begin their walk over K at 0
            assert torch.equal(out[lo:lo + n, :512], api.gemm_tiles(x[lo:lo + n].clone(), w[g])[:, :512]), g
        lo += n
    rows = sum(counts) - 1                                              # the same bits, whichever tile: of the last group as if it were alone
    alone = api.gemm_mfma_grouped(x[rows:].contiguous(), w[-1:].contiguous(), torch.tensor([0, 1], dtype=torch.int32, device=DEV))
    assert torch.equal(alone[0], out[rows])
