"""Prompt attention with 32 rows of a head a wave (csrc/attention_prefill.h) at the edges of its tiles, against the plain kernel and
plain attention in 64 bits."""
import math

import pytest
import torch

pytestmark = pytest.mark.gpu
DEV = "cuda"
D = 128


def K():
    from infernum_amd.kernels import api
    return api


def _case(nh, nkv, ps, lens, q_lens, seed, cols=None, poison=True, D=D):
    """Requests of lens keys whose last q_lens tokens are new, pages in a shuffled order; what no request holds is NaN."""
    g = torch.Generator(device=DEV).manual_seed(seed)
    rnd = lambda *s: torch.randn(*s, device=DEV, generator=g).to(torch.bfloat16)                     # noqa: E731
    counts = [-(-n // ps) for n in lens]
    P = sum(counts) + 2
    order = torch.randperm(P - 1, device=DEV, generator=g).int() + 1
    bt = torch.full((len(lens), cols or max(counts)), 0, dtype=torch.int32, device=DEV)
    kp = torch.full((P, nkv, ps, D), float("nan") if poison else 0.0, dtype=torch.bfloat16, device=DEV)
    vp = torch.full((P, nkv, D, ps), float("nan") if poison else 0.0, dtype=torch.bfloat16, device=DEV)
    k = [rnd(n, nkv, D) for n in lens]
    v = [rnd(n, nkv, D) for n in lens]
    at = 0
    for i, n in enumerate(lens):
        bt[i, :counts[i]] = order[at:at + counts[i]]
        at += counts[i]
        for p in range(counts[i]):
            page, a, b = int(bt[i, p]), p * ps, min(n, p * ps + ps)
            kp[page, :, :b - a] = k[i][a:b].transpose(0, 1)
            vp[page, :, :, :b - a] = v[i][a:b].permute(1, 2, 0)
    q = rnd(sum(q_lens), nh * D)
    i32 = lambda x: torch.tensor(x, dtype=torch.int32, device=DEV)                                   # noqa: E731
    starts = i32([sum(q_lens[:i]) for i in range(len(q_lens) + 1)])
    ctx = i32([a - b for a, b in zip(lens, q_lens)])
    tiles = i32([(s, r) for s in range(len(lens)) for r in range(0, q_lens[s], 64)]).reshape(-1, 2)
    return dict(q=q, k=k, v=v, kp=kp, vp=vp, bt=bt, starts=starts, ctx=ctx, tiles=tiles, lens=lens, q_lens=q_lens)


def _run(c, nh, nkv, window=0, **kw):
    out = torch.full_like(c["q"], float("nan"))
    D = c["kp"].shape[3]
    K().attention_prefill(c["q"], c["kp"], c["vp"], out, c["starts"], c["ctx"], c["bt"], c["tiles"], c["tiles"].shape[0], nh, nkv, D,
                          D ** -0.5, window, **kw)
    return out


def _want(c, nh, nkv, window):
    rows, at = [], 0
    D = c["kp"].shape[3]
    for k, v, n, m in zip(c["k"], c["v"], c["lens"], c["q_lens"]):
        q = c["q"][at:at + m].view(m, nh, D).double()
        at += m
        pos, key = torch.arange(n - m, n, device=DEV)[:, None], torch.arange(n, device=DEV)[None, :]
        first = pos - window + 1 if window > 0 else pos // -window * -window if window < 0 else 0      # < 0: chunks of -window keys
        seen = (key <= pos) & (key >= first)
        for_heads = lambda t: t.double().repeat_interleave(nh // nkv, dim=1)                         # noqa: E731
        s = torch.einsum("qhd,khd->hqk", q, for_heads(k)) * D ** -0.5
        p = torch.softmax(s.masked_fill(~seen, -math.inf), dim=-1)
        rows.append(torch.einsum("hqk,khd->qhd", p, for_heads(v)).reshape(m, nh * D))
    return torch.cat(rows)


@pytest.mark.parametrize("nh,nkv,ps", [(4, 1, 16), (6, 2, 8), (4, 2, 64), (14, 2, 32), (8, 2, 128)])
@pytest.mark.parametrize("lens,q_lens", [([1, 2, 31, 32, 33], [1, 2, 31, 32, 33]), ([63, 64, 65, 127, 129], [63, 64, 65, 127, 129]),
                                         ([95, 96, 97, 200, 161], [1, 33, 65, 64, 7]), ([300, 449], [300, 100])])
@pytest.mark.parametrize("window", [0, 1, 40, 100])
def test_edges_of_tiles(nh, nkv, ps, lens, q_lens, window):
    c = _case(nh, nkv, ps, lens, q_lens, seed=nh * ps + len(lens) + window)
    out = _run(c, nh, nkv, window)
    # probabilities within 2^-9 of themselves (their sum is taken of the rounded ones), values of order one, one rounding to bf16
    err = (out.double() - _want(c, nh, nkv, window)).abs().max().item()
    assert err <= 2.5e-2, err
    for hpw in (1, 2, 4):
        for paired in (False, True):
            assert torch.equal(_run(c, nh, nkv, window, heads_per_workgroup=hpw, paired=paired), out), (hpw, paired)
    # a wide block table takes the kernel with 16 rows a wave: as near
    wide = _case(nh, nkv, ps, lens, q_lens, seed=nh * ps + len(lens) + window, cols=4097)
    assert ((_run(wide, nh, nkv, window).double() - out.double()).abs().max().item()) <= 2.5e-2


def test_whole_and_in_portions_the_same_bits():
    nh, nkv, ps, n = 8, 2, 16, 333
    whole = _case(nh, nkv, ps, [n], [n], seed=3)
    want = _run(whole, nh, nkv)
    for a, b in ((0, 64), (64, 100), (100, 333), (31, 32), (200, 333)):
        part = dict(whole, q=whole["q"][a:b].clone(), lens=[b], q_lens=[b - a], ctx=torch.tensor([a], dtype=torch.int32, device=DEV),
                    starts=torch.tensor([0, b - a], dtype=torch.int32, device=DEV),
                    tiles=torch.tensor([(0, r) for r in range(0, b - a, 64)], dtype=torch.int32, device=DEV).reshape(-1, 2))
        assert torch.equal(_run(part, nh, nkv), want[a:b]), (a, b)


def test_a_later_token_that_is_not_finite_stays_out_of_the_rows_before_it():
    """Keys and values of a token are read by workgroups whose earlier rows do not see it."""
    nh, nkv, ps, n = 4, 1, 16, 200
    for bad in (float("inf"), float("nan")):
        c = _case(nh, nkv, ps, [n], [n], seed=4)
        want = _run(c, nh, nkv)
        t = 170                                                         # its half of a tile begins at key 160
        page = int(c["bt"][0, t // ps])
        c["kp"][page, :, t % ps] = bad
        got = _run(c, nh, nkv)
        assert torch.equal(got[:t], want[:t])
        c["vp"][page, :, :, t % ps] = bad
        got = _run(c, nh, nkv)
        assert torch.equal(got[:160], want[:160]) and not bool(got[t:].isfinite().all())


def test_a_key_without_a_page_gives_nan():
    nh, nkv, ps = 4, 1, 16
    c = _case(nh, nkv, ps, [100, 64], [100, 64], seed=5)
    c["bt"][0, 2] = -1
    out = _run(c, nh, nkv)
    assert bool(out[64:100].isnan().all()) and bool(out[100:].isfinite().all())
    c["bt"][0, 2] = 10 ** 6
    assert bool(_run(c, nh, nkv)[64:100].isnan().all())


@pytest.mark.parametrize("nh,nkv,ps", [(4, 1, 16), (6, 2, 8), (4, 2, 64)])
@pytest.mark.parametrize("lens,q_lens", [([1, 31, 33, 64, 129], [1, 31, 33, 64, 129]), ([300, 449], [300, 100])])
@pytest.mark.parametrize("window", [0, 40, -96])
def test_the_block_tables_width_leaves_the_bits_alone(nh, nkv, ps, lens, q_lens, window):
    """A neighbour's length makes a step's tables wider than the kernel keeps in LDS: the other kernel, the same order of sums."""
    c = _case(nh, nkv, ps, lens, q_lens, seed=nh + ps + len(lens))
    out = _run(c, nh, nkv, window)
    c["bt"] = torch.cat([c["bt"], torch.zeros(len(lens), 4097, dtype=torch.int32, device=DEV)], dim=1).contiguous()
    for hpw in (1, 2, 4):
        for paired in (False, True):
            assert torch.equal(_run(c, nh, nkv, window, heads_per_workgroup=hpw, paired=paired), out), (hpw, paired)


def _first_visible(pos, window):
    return 0 if window == 0 else max(0, pos - window + 1) if window > 0 else pos // -window * -window


@pytest.mark.parametrize("ctx,n,window", [(16, 100, 0), (1, 64, 0), (15, 97, 0), (17, 97, 0), (0, 200, 40), (16, 200, 33), (5, 150, 1),
                                          (40, 130, 100), (0, 200, -48), (30, 170, -128), (0, 257, -16)])
def test_a_value_that_is_not_finite_reaches_the_16_rows_that_meet_its_32_keys(ctx, n, window):
    """A key's half of a tile is weighed in for a block of 16 rows if one of them may see a key of it; no other row may change."""
    nh, nkv, ps, total = 4, 1, 16, ctx + n
    c = _case(nh, nkv, ps, [total], [n], seed=9)
    wide = dict(c, bt=torch.cat([c["bt"], torch.zeros(1, 4097, dtype=torch.int32, device=DEV)], dim=1).contiguous())
    want = _run(c, nh, nkv, window)
    assert bool(want.isfinite().all())
    for t in sorted({0, 15, 31, 32, 40, 63, 64, 95, 100, ctx, total - 1}):
        if t >= total:
            continue
        page = int(c["bt"][0, t // ps])
        was = c["vp"][page, :, :, t % ps].clone()
        c["vp"][page, :, :, t % ps] = float("inf")
        meets = torch.zeros(n, dtype=torch.bool, device=DEV)
        for first in range(0, n, 16):
            lo, hi = _first_visible(ctx + first, window), ctx + min(first + 15, n - 1)
            meets[first:first + 16] = lo // 32 <= t // 32 <= hi // 32
        sees = torch.tensor([_first_visible(ctx + r, window) <= t <= ctx + r for r in range(n)], device=DEV)
        for case, paired in ((c, False), (c, True), (wide, False)):
            got = _run(case, nh, nkv, window, paired=paired)
            assert torch.equal(got[~meets], want[~meets]), (t, paired)
            assert not bool(got[sees].isfinite().any()), (t, paired)
        c["vp"][page, :, :, t % ps] = was


def test_short_ranges_of_keys_go_to_waves_of_16_rows():
    """Where the line lies, and the same bits on both sides of it, through the shape that a step's launch is given."""
    api = K()
    dev = torch.device(DEV)
    cus = torch.cuda.get_device_properties(dev).multi_processor_count
    of_two, of_four = api.PREFILL_NARROW_KEYS
    narrow = lambda q, c, nh=32, nkv=8, w=0, d=128: bool(api.prefill_shape(nh, nkv, d, q, c, w, dev) & api.PREFILL_NARROW)    # noqa: E731
    assert narrow([20], [0]) and narrow([64], [of_two - 64]) and not narrow([64], [of_two - 63])
    assert narrow([64] * cus, [of_four - 64] * cus) and not narrow([64] * cus, [of_four - 63] * cus)
    assert narrow([64], [5000], w=500) and not narrow([64], [5000], w=2000)
    chunk = api.PREFILL_NARROW_CHUNK
    assert narrow([64], [5000], w=-chunk) and not narrow([64], [5000], w=-chunk - 1) and not narrow([64], [5024], w=-chunk)
    assert narrow([64], [5024], w=-500)
    assert not narrow([20], [0], nh=8) and not narrow([20], [0], d=64) and not narrow([], [])
    for window in (0, 100, -64):
        c = _case(8, 2, 16, [200, 33], [120, 33], seed=11)
        shape = api.prefill_shape(8, 2, D, c["q_lens"], [80, 0], window, dev)
        assert shape & api.PREFILL_NARROW
        want = _run(c, 8, 2, window)
        assert torch.equal(_run(c, 8, 2, window, heads_per_workgroup=shape), want)
        assert torch.equal(_run(c, 8, 2, window, heads_per_workgroup=shape & ~api.PREFILL_NARROW), want)
    with pytest.raises(api.KernelError):
        _run(c, 8, 2, heads_per_workgroup=0x402)


@pytest.mark.parametrize("nh,nkv,ps", [(4, 1, 16), (6, 2, 8), (4, 2, 64)])
@pytest.mark.parametrize("lens,q_lens", [([1, 2, 31, 32, 33], [1, 2, 31, 32, 33]), ([95, 96, 97, 200, 161], [1, 33, 65, 64, 7]),
                                         ([300, 449], [300, 100])])
@pytest.mark.parametrize("chunk", [1, 16, 48, 64, 100, 300])
def test_chunks_at_the_edges_of_tiles(nh, nkv, ps, lens, q_lens, chunk):
    c = _case(nh, nkv, ps, lens, q_lens, seed=nh * ps + len(lens) + chunk)
    rows, at = [], 0
    for k, v, n, m in zip(c["k"], c["v"], c["lens"], c["q_lens"]):
        q = c["q"][at:at + m].view(m, nh, D).double()
        at += m
        pos, key = torch.arange(n - m, n, device=DEV)[:, None], torch.arange(n, device=DEV)[None, :]
        s = torch.einsum("qhd,khd->hqk", q, k.double().repeat_interleave(nh // nkv, dim=1)) * D ** -0.5
        p = torch.softmax(s.masked_fill((key > pos) | (key < pos // chunk * chunk), -math.inf), dim=-1)
        rows.append(torch.einsum("hqk,khd->qhd", p, v.double().repeat_interleave(nh // nkv, dim=1)).reshape(m, nh * D))
    want = torch.cat(rows)
    first = _run(c, nh, nkv, -chunk)
    # as above: probabilities within 2^-9 of themselves, values of order one (a chunk of one key: of up to 4.5), one rounding to bf16
    assert ((first.double() - want).abs() <= 1.5e-2 + 2.0 ** -8 * want.abs()).all(), (first.double() - want).abs().max().item()
    for hpw in (1, 2, 4, K().PREFILL_NARROW | 2):
        assert torch.equal(_run(c, nh, nkv, -chunk, heads_per_workgroup=hpw), first), hpw


@pytest.mark.parametrize("lens,q_lens", [([1, 2, 31, 32, 33], [1, 2, 31, 32, 33]), ([95, 200, 161], [1, 64, 7]), ([300, 449], [300, 100])])
@pytest.mark.parametrize("window", [0, 40])
def test_sinks_and_rows_that_lie_apart(lens, q_lens, window):
    """A sink takes its share of every row's probabilities; queries and results as column ranges of wider rows."""
    nh, nkv, ps = 8, 2, 16
    c = _case(nh, nkv, ps, lens, q_lens, seed=21)
    sinks = torch.linspace(-3.0, 6.0, nh, device=DEV)
    rows, at = [], 0
    for k, v, n, m in zip(c["k"], c["v"], c["lens"], c["q_lens"]):
        q = c["q"][at:at + m].view(m, nh, D).double()
        at += m
        pos, key = torch.arange(n - m, n, device=DEV)[:, None], torch.arange(n, device=DEV)[None, :]
        s = torch.einsum("qhd,khd->hqk", q, k.double().repeat_interleave(nh // nkv, dim=1)) * D ** -0.5
        s = s.masked_fill((key > pos) | ((key <= pos - window) if window else (key < 0)), -math.inf)
        p = torch.softmax(torch.cat([s, sinks.double()[:, None, None].expand(nh, m, 1)], dim=2), dim=-1)[:, :, :-1]
        rows.append(torch.einsum("hqk,khd->qhd", p, v.double().repeat_interleave(nh // nkv, dim=1)).reshape(m, nh * D))
    first = _run(c, nh, nkv, window, sinks=sinks)
    assert (first.double() - torch.cat(rows)).abs().max().item() <= 2.5e-2
    assert torch.equal(_run(c, nh, nkv, window, sinks=sinks, heads_per_workgroup=K().PREFILL_NARROW | 4), first)
    wide_q = torch.full((c["q"].shape[0], nh * D + 2 * nkv * D), float("nan"), dtype=torch.bfloat16, device=DEV)
    wide_q[:, :nh * D] = c["q"]
    wide_o = torch.full((c["q"].shape[0], nh * D + 64), 7.0, dtype=torch.bfloat16, device=DEV)
    K().attention_prefill(wide_q[:, :nh * D], c["kp"], c["vp"], wide_o[:, :nh * D], c["starts"], c["ctx"], c["bt"], c["tiles"],
                          c["tiles"].shape[0], nh, nkv, D, D ** -0.5, window, sinks=sinks)
    assert torch.equal(wide_o[:, :nh * D], first) and bool((wide_o[:, nh * D:] == 7.0).all())


@pytest.mark.parametrize("nh,nkv,ps", [(4, 1, 16), (6, 2, 8), (3, 1, 64)])
@pytest.mark.parametrize("lens,q_lens", [([1, 2, 31, 32, 33], [1, 2, 31, 32, 33]), ([63, 64, 65, 127, 129], [63, 64, 65, 127, 129]),
                                         ([95, 96, 97, 200, 161], [1, 33, 65, 64, 7]), ([300, 449], [300, 100])])
@pytest.mark.parametrize("window", [0, 1, 40, 100, -16, -48, -96])
def test_heads_of_256_at_the_edges_of_tiles(nh, nkv, ps, lens, q_lens, window):
    """A tile is one half of 32 keys there: the kernel's other loop, and the same bits from waves of 16 rows."""
    c = _case(nh, nkv, ps, lens, q_lens, seed=nh * ps + len(lens) + window, D=256)
    first = _run(c, nh, nkv, window, heads_per_workgroup=K().PREFILL_NARROW | 2)
    want = _want(c, nh, nkv, window)     # as for heads of 128 above: windows, and chunks
    assert ((first.double() - want).abs() <= (2.5e-2 if window >= 0 else 1.5e-2 + 2.0 ** -8 * want.abs())).all()
    for hpw in (0, 1, 2):
        for paired in (False, True):
            assert torch.equal(_run(c, nh, nkv, window, heads_per_workgroup=hpw, paired=paired), first), (hpw, paired)
    with pytest.raises(K().KernelError):
        _run(c, nh, nkv, window, heads_per_workgroup=4)
    t, page = lens[-1] - 1, int(c["bt"][-1, (lens[-1] - 1) // ps])              # a value that the rows before its 16 do not meet
    c["vp"][page, :, :, t % ps] = float("inf")
    bad, other = _run(c, nh, nkv, window), _run(c, nh, nkv, window, heads_per_workgroup=K().PREFILL_NARROW | 2)
    finite = bad.isfinite()              # the same rows from both kernels (infinite or NaN is up to each), and the same bits elsewhere
    assert torch.equal(finite, other.isfinite()) and torch.equal(bad[finite], other[finite])
    blocks = -(-q_lens[-1] // 16) - 1
    clean = [r for r in range(blocks * 16) if (lens[-1] - q_lens[-1] + r // 16 * 16 + 15) // 32 < t // 32]
    assert torch.equal(bad[bad.shape[0] - q_lens[-1]:][clean], first[first.shape[0] - q_lens[-1]:][clean]) and not bool(bad[-1].isfinite().any())


@pytest.mark.parametrize("ctx,n,window", [(16, 100, 0), (1, 64, 0), (17, 97, 0), (0, 200, 40), (16, 200, 33), (5, 150, 1), (40, 130, 100),
                                          (0, 200, -48), (30, 170, -128), (0, 257, -16)])
def test_heads_of_256_and_a_value_that_is_not_finite(ctx, n, window):
    """It reaches blocks of 16 rows that meet its 32 keys, the same in both kernels, and no other row."""
    nh, nkv, ps, total = 4, 1, 16, ctx + n
    c = _case(nh, nkv, ps, [total], [n], seed=9, D=256)
    want = _run(c, nh, nkv, window)
    assert bool(want.isfinite().all())
    for t in sorted({0, 15, 31, 32, 40, 63, 64, 95, 100, ctx, total - 1}):
        if t >= total:
            continue
        page = int(c["bt"][0, t // ps])
        was = c["vp"][page, :, :, t % ps].clone()
        c["vp"][page, :, :, t % ps] = float("inf")
        meets = torch.zeros(n, dtype=torch.bool, device=DEV)
        for first in range(0, n, 16):
            lo, hi = _first_visible(ctx + first, window), ctx + min(first + 15, n - 1)
            meets[first:first + 16] = lo // 32 <= t // 32 <= hi // 32
        sees = torch.tensor([_first_visible(ctx + r, window) <= t <= ctx + r for r in range(n)], device=DEV)
        for paired in (False, True):     # (a key behind the last that a workgroup's rows see is nobody's there)
            got, other = (_run(c, nh, nkv, window, heads_per_workgroup=shape, paired=paired) for shape in (2, K().PREFILL_NARROW | 2))
            assert torch.equal(got[~meets], want[~meets]) and not bool(got[sees].isfinite().any()), (t, paired)
            finite = got.isfinite()
            assert torch.equal(finite, other.isfinite()) and torch.equal(got[finite], other[finite]), (t, paired)
        c["vp"][page, :, :, t % ps] = was


@pytest.mark.parametrize("lens,q_lens", [([1, 2, 31, 32, 33], [1, 2, 31, 32, 33]), ([300, 449], [300, 100])])
@pytest.mark.parametrize("window", [0, 40])
def test_heads_of_256_with_sinks(lens, q_lens, window):
    nh, nkv, ps = 4, 1, 16
    c = _case(nh, nkv, ps, lens, q_lens, seed=23, D=256)
    sinks = torch.linspace(-3.0, 6.0, nh, device=DEV)
    first = _run(c, nh, nkv, window, sinks=sinks)
    rows, at = [], 0                     # a sink leaves of a row what the keys' part of its denominator is
    for k, n, m in zip(c["k"], c["lens"], c["q_lens"]):
        q = c["q"][at:at + m].view(m, nh, 256).transpose(0, 1).double()
        at += m
        pos, key = torch.arange(n - m, n, device=DEV)[:, None], torch.arange(n, device=DEV)[None, :]
        s = torch.matmul(q, k.double().permute(1, 2, 0).contiguous()) * 256 ** -0.5
        total = s.masked_fill((key > pos) | ((key <= pos - window) if window else (key < 0)), -math.inf).logsumexp(dim=-1)
        rows.append(torch.sigmoid(total - sinks.double()[:, None]).t().repeat_interleave(256, dim=1))
    assert (first.double() - _want(c, nh, nkv, window) * torch.cat(rows)).abs().max().item() <= 2.5e-2
    for shape in (1, K().PREFILL_NARROW | 2):
        assert torch.equal(_run(c, nh, nkv, window, sinks=sinks, heads_per_workgroup=shape), first), shape


@pytest.mark.parametrize("nh,nkv,ps", [(4, 1, 16), (6, 2, 8)])
@pytest.mark.parametrize("lens,q_lens", [([1, 31, 33, 64, 129], [1, 31, 33, 64, 129]), ([300, 449], [300, 100])])
@pytest.mark.parametrize("window", [0, 40, -96])
def test_heads_of_256_sum_in_the_order_of_a_head_alone(nh, nkv, ps, lens, q_lens, window):
    """Heads that share keys, in either kernel, leave the bits that each leaves with keys of its own (a launch that has one kernel alone)."""
    c = _case(nh, nkv, ps, lens, q_lens, seed=nh * ps + len(lens) + window, D=256)
    own = dict(c, kp=c["kp"].repeat_interleave(nh // nkv, dim=1).contiguous(), vp=c["vp"].repeat_interleave(nh // nkv, dim=1).contiguous())
    want = _run(own, nh, nh, window)
    for shape in (1, 2, K().PREFILL_NARROW | 1, K().PREFILL_NARROW | 2):
        assert torch.equal(_run(c, nh, nkv, window, heads_per_workgroup=shape), want), shape


def test_short_ranges_of_heads_of_256_go_to_waves_of_16_rows():
    api, dev = K(), torch.device(DEV)
    narrow = lambda q, c, nh=16, nkv=1, w=0: bool(api.prefill_shape(nh, nkv, 256, q, c, w, dev) & api.PREFILL_NARROW)    # noqa: E731
    line = api.PREFILL_NARROW_KEYS_256
    assert narrow([line], [0]) and not narrow([line + 1], [0]) and narrow([30], [line - 30]) and not narrow([30], [line - 29])
    assert narrow([64], [5000], w=line - 64) and not narrow([64], [5000], w=line - 63) and not narrow([20], [0], nh=1)
    assert narrow([64], [5000], w=-1024) and not narrow([64], [5024], w=-1024) and not narrow([64], [5000], w=-api.PREFILL_NARROW_CHUNK - 1)
