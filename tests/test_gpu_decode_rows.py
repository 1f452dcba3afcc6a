"""GPU: the many-row kernel (more than 16 query rows per KV head, decode_rows.h) against the oracle.

Sizes sit at the edges of its tiles (32, 64, 128 and 256 rows), chunks (128 tokens) and pages. bf16 results at the decode
tolerance; float32 results within 2^-14 of the largest output: the value weights carry at least 22 bits, so what is
left is the float32 rounding of scores up to 2^7 base-2 units (2^-18 each, on both sides: a weight off by up to
2^-17 ln 2 in the kernel and in the oracle, times the few that accumulate).
"""

import numpy as np
import pytest
import torch

from test_gpu_decode import DEV, check, make_case, run_case

pytestmark = pytest.mark.gpu

FORMATS = [("fp8", "head"), ("int8", "token"), ("bf16", None), ("int8", "head"), ("fp8", "token")]


@pytest.mark.parametrize("fmt,scales", FORMATS)
@pytest.mark.parametrize("nq,hq,hkv", [(17, 4, 4), (16, 4, 2), (11, 6, 2), (32, 4, 2), (13, 10, 2), (64, 2, 1), (43, 3, 1), (150, 4, 2)])
def test_rows_at_tile_edges(fmt, scales, nq, hq, hkv):
    c = make_case(fmt, [517, 0, nq, 128, 129, 1, 260], hq=hq, hkv=hkv, nq=nq, scales=scales, seed=nq)
    got, want = run_case(c)
    check(got, want, f"{fmt}/{scales} {nq} queries, {hq}/{hkv} heads")
    assert got[1].float().abs().sum().item() == 0  # no tokens: zeros


def longer_bound(c, context=8192):
    """The case with block tables for `context` tokens: calls bounded by that take the tiles of a large call."""
    page = c["k"].shape[1]
    return dict(c, table=torch.nn.functional.pad(c["table"], (0, context // page - c["table"].shape[1])))


@pytest.mark.parametrize("fmt,scales", FORMATS)
@pytest.mark.parametrize("nq,hq,hkv,tile", [(16, 4, 2, 32), (11, 6, 2, 64), (32, 4, 2, 64), (13, 10, 2, 128), (64, 2, 1, 128), (43, 3, 1, 128), (150, 4, 2, 128)])
def test_rows_at_tile_edges_under_a_longer_bound(fmt, scales, nq, hq, hkv, tile):
    """The same edges in the tiles that large calls take: a bound on the lengths far above them (their own bound would give
    32- or 64-row tiles)."""
    from bpt_amd import decode_plan

    c = longer_bound(make_case(fmt, [517, 0, nq, 128, 129, 1, 260], hq=hq, hkv=hkv, nq=nq, scales=scales, seed=nq))
    plan = decode_plan(c["q"], c["k"], c["v"], c["table"], c["lens"], c["ks"], c["vs"], scale=0.1, max_context=8192)
    assert plan[1] == 128 and plan[2] == -(-2 * plan[0] * tile * 129 * 4 // 256) * 256
    got, want = run_case(c, max_context=8192)
    check(got, want, f"{fmt}/{scales} {nq} queries, {hq}/{hkv} heads")


@pytest.mark.parametrize("fmt,scales", FORMATS)
@pytest.mark.parametrize("page", [1, 2, 8, 16, 128])
@pytest.mark.parametrize("q_dtype", [torch.bfloat16, torch.float16])
def test_rows_page_sizes_and_q_dtypes(fmt, scales, page, q_dtype):
    c = make_case(fmt, [300, 77], hq=8, hkv=2, nq=9, page=page, scales=scales, seed=page, table_dtype=torch.int64)
    got, want = run_case(c, q=c["q"].to(q_dtype), out_dtype=q_dtype)
    check(got, want, f"{fmt}/{scales} page {page} {q_dtype}")


@pytest.mark.parametrize("fmt,scales", FORMATS)
@pytest.mark.parametrize("nq,q_dtype", [(256, torch.bfloat16), (257, torch.float16), (300, torch.bfloat16)])
def test_rows_wide_tiles(fmt, scales, nq, q_dtype):
    """256-row tiles, pieces combined by the second launch: 1024 rows per KV head are four whole tiles, 1028 and 1200
    leave a part of one; sequences of no tokens, of the new ones alone and of some more."""
    from bpt_amd import decode_plan

    c = make_case(fmt, [2900, 0, nq, 700], hq=32, hkv=8, nq=nq, scales=scales, seed=nq)
    plan = decode_plan(c["q"], c["k"], c["v"], c["table"], c["lens"], c["ks"], c["vs"], scale=0.1, max_context=2900)
    assert plan[2] >= 2 * plan[0] * 256 * 129 * 4  # 256-row slots
    got, want = run_case(c, q=c["q"].to(q_dtype), out_dtype=q_dtype)
    check(got, want, f"{fmt}/{scales} {nq} queries {q_dtype}")


@pytest.mark.parametrize("nq", [40, 100])
def test_rows_two_launches_replay_in_a_graph(nq):
    """Both launches under capture, replayed with eager work between: the partials of one replay are not the next's."""
    from bpt_amd import paged_decode_attention

    c = make_case("fp8", [3000, 450], hq=16, hkv=2, nq=nq, seed=nq)
    args = (c["q"], c["k"], c["v"], c["table"], c["lens"], c["ks"], c["vs"])
    want = paged_decode_attention(*args, scale=0.09, max_context=3000)
    out = torch.empty_like(want)
    stream = torch.cuda.Stream()
    with torch.cuda.stream(stream):
        paged_decode_attention(*args, scale=0.09, max_context=3000, out=out)
    torch.cuda.synchronize()
    graph = torch.cuda.CUDAGraph()
    with torch.cuda.graph(graph, stream=stream):
        paged_decode_attention(*args, scale=0.09, max_context=3000, out=out)
    for _ in range(3):
        out.zero_()
        graph.replay()
        torch.cuda.synchronize()
        assert torch.equal(out, want)
        paged_decode_attention(*args, scale=0.09, max_context=3000)
        torch.cuda.synchronize()


def test_rows_two_launches_timed():
    """The timed entry point over a call of two launches: the start event on the first, the stop event on the second."""
    from bpt_amd import paged_decode_attention

    c = make_case("fp8", [3000, 450], hq=16, hkv=2, nq=100, seed=100)
    args = (c["q"], c["k"], c["v"], c["table"], c["lens"], c["ks"], c["vs"])
    want = paged_decode_attention(*args, scale=0.09, max_context=3000)
    start, mid, stop, end = (torch.cuda.Event(enable_timing=True) for _ in range(4))
    for e in (start, mid, stop, end):
        e.record()
    torch.cuda.synchronize()
    start.record()
    got = paged_decode_attention(*args, scale=0.09, max_context=3000, _events=(mid.cuda_event, stop.cuda_event))
    end.record()
    torch.cuda.synchronize()
    assert torch.equal(got, want)
    assert 0 < mid.elapsed_time(stop) <= start.elapsed_time(end)


@pytest.mark.parametrize("num_splits", [1, 3, 1000])
@pytest.mark.parametrize("nq", [10, 20, 40])
def test_rows_forced_splits(num_splits, nq):
    c = make_case("fp8", [2000, 131, 40], hq=8, hkv=2, nq=nq, seed=num_splits)
    got, want = run_case(c, num_splits=num_splits)
    check(got, want, f"{nq} queries, {num_splits} splits")


@pytest.mark.parametrize("fmt,scales", FORMATS)
@pytest.mark.parametrize("nq,q_dtype", [(10, torch.bfloat16), (20, torch.float16), (40, torch.bfloat16)])
def test_rows_long_context_in_float32(fmt, scales, nq, q_dtype):
    c = make_case(fmt, [9000, 700], hq=8, hkv=2, nq=nq, scales=scales, seed=nq, head_major=True)
    got, want = run_case(c, q=c["q"].to(q_dtype), out_dtype=torch.float32)
    err = np.abs(got.cpu().numpy() - want).max()
    assert err <= 2.0**-14 * np.abs(want).max(), f"{fmt}/{scales}: {err:.3e}"


def test_rows_negative_scale_and_lse_and_repeats():
    from bpt_amd import paged_decode_attention
    from oracle import attention
    from test_gpu_decode import np_codes

    c = make_case("fp8", [900, 33], hq=8, hkv=2, nq=12, seed=5)
    lse = torch.empty((2, 12, 8), device=DEV)
    args = (c["q"], c["k"], c["v"], c["table"], c["lens"], c["ks"], c["vs"])
    got = paged_decode_attention(*args, scale=-0.05, max_context=900, lse=lse, out_dtype=torch.float32)
    again = paged_decode_attention(*args, scale=-0.05, max_context=900, out_dtype=torch.float32)
    want, want_lse = attention.paged_decode(
        c["q"].float().cpu().numpy(), np_codes(c["k"], "fp8"), np_codes(c["v"], "fp8"), c["table"].cpu().numpy(),
        c["lens"].cpu().numpy(), c["ks"].cpu().numpy(), c["vs"].cpu().numpy(), "fp8", -0.05)
    assert torch.equal(got, again)
    assert np.abs(got.cpu().numpy() - want).max() <= 2.0**-14 * np.abs(want).max()
    seen = np.isfinite(want_lse)
    assert np.array_equal(np.isfinite(lse.cpu().numpy()), seen)
    assert np.abs(lse.cpu().numpy() - want_lse)[seen].max() < 1e-4


@pytest.mark.parametrize("q_dtype", [torch.bfloat16, torch.float16])
@pytest.mark.parametrize("context", [64, 8192])  # the second takes tiles of up to 256 rows
@pytest.mark.parametrize("hq,nq", [(17, 1), (33, 1), (65, 1), (300, 1), (64, 40)])
def test_rows_int8_weights_keep_all_24_bits(hq, nq, q_dtype, context):
    """One visible token with zero keys: its weight is 2^4 times its float32 value scale, so a code that is a power of two
    gives that scale times the code exactly, if the weight keeps its 24 bits and its exponent (2^-60 .. 2^90)."""
    from bpt_amd import paged_decode_attention

    g = torch.Generator(device=DEV).manual_seed(hq)
    b, t, hkv = 40, nq, 1
    k = torch.zeros((b, 16 * 4, hkv, 128), dtype=torch.int8, device=DEV).view(b * 4, 16, hkv, 128)
    codes = torch.tensor([1, 2, -4, 64, -128], dtype=torch.int8, device=DEV)
    v = codes[torch.randint(5, k.shape, generator=g, device=DEV)]
    vs = (torch.rand(k.shape[:3], generator=g, device=DEV) + 1) * torch.exp2(torch.randint(-60, 91, k.shape[:3], generator=g, device=DEV).float())
    ks = torch.ones_like(vs)
    table = torch.zeros((b, context // 16), dtype=torch.int32, device=DEV)
    table[:, :4] = torch.arange(b * 4, dtype=torch.int32, device=DEV).view(b, 4)
    lens = torch.full((b,), t, dtype=torch.int32, device=DEV)
    q = torch.randn((b, nq, hq, 128), generator=g, device=DEV).to(q_dtype)
    got = paged_decode_attention(q, k, v, table, lens, ks, vs, scale=0.1, max_context=context, out_dtype=torch.float32)
    want = v.view(b, 64, 128)[:, 0].float() * vs.view(b, 64)[:, :1]
    assert torch.equal(got[:, 0], want[:, None].expand(b, hq, 128))  # the first query sees the first token alone


def test_rows_int8_scales_over_the_float32_range():
    """Value scales of 0 and from 2^-40 to 2^80 in one sequence, against the oracle: float32 within 2^-14 of the largest."""
    c = make_case("int8", [700, 90], hq=64, hkv=2, nq=2, scales="token", seed=3)
    g = torch.Generator(device=DEV).manual_seed(4)
    for lo, hi in ((70, 81), (-40, -29), (-40, 81)):
        e = torch.randint(lo, hi, c["vs"].shape, generator=g, device=DEV).float()
        d = dict(c, vs=torch.where(torch.rand(e.shape, generator=g, device=DEV) < 0.2, 0.0, c["vs"] * torch.exp2(e)))
        got, want = run_case(d, out_dtype=torch.float32)
        err = np.abs(got.cpu().numpy() - want).max()
        assert err <= 2.0**-14 * np.abs(want).max(), f"2^{lo} .. 2^{hi}: {err:.3e}"


def plant_nonfinite(c, nq, with_stale=True):
    """Values (BF16), NaN codes (FP8) or value scales (per token) that are not finite, at a token that every query sees, at
    several of the new ones and at each sequence's last. Returns the oracle's pools, those at zero, and the planted values
    as [(sequence, token, head, 128 values)]. with_stale: every slot that holds no token becomes NaN too."""
    fmt, per_token = c["fmt"], c["vs"] is not None and c["vs"].dim() == 3
    k, v, lens, page = c["k"], c["v"].clone(), c["lens"].tolist(), c["k"].shape[1]
    ks, vs = (None if x is None else x.clone() for x in (c["ks"], c["vs"]))
    raw = v if fmt != "fp8" else v.view(torch.uint8)
    slot = lambda b, t: (int(c["table"][b, t // page]), t % page)  # noqa: E731
    if with_stale:
        used = torch.zeros(v.shape[:2], dtype=torch.bool, device=DEV)
        for b, n in enumerate(lens):
            at = torch.arange(n, device=DEV)
            used[c["table"][b, at // page].long(), at % page] = True
        if fmt != "int8":
            raw[~used] = float("nan") if fmt == "bf16" else 0x7F
            k = k.clone()
            (k if fmt == "bf16" else k.view(torch.uint8))[~used] = float("nan") if fmt == "bf16" else 0xFF
        if per_token:
            ks[~used], vs[~used] = float("nan"), float("nan")
    clean_v, clean_vs, planted = v.clone(), None if vs is None else vs.clone(), []
    heads = v.shape[2]
    for b, n in enumerate(lens):
        for i, t in enumerate(sorted({0 if b % 2 else n // 3, n - nq + 3, n - nq // 2, n - 2, n - 1})):
            if not 0 <= t < n:
                continue
            h, ch, (e, o) = (b + i) % heads, 31 * (b + i) % 128, slot(b, t)
            bad = torch.zeros(128)
            if per_token:
                x = [float("inf"), float("nan"), float("-inf")][i % 3]
                bad = (v[e, o, h].float() * x).cpu()
                vs[e, o, h], clean_vs[e, o, h] = x, 0.0
            else:
                for j, x in enumerate([float("inf"), float("-inf"), float("nan")] if fmt == "bf16" else [float("nan")] * 3):
                    bad[(ch + j) % 128] = x
                    raw[e, o, h, (ch + j) % 128] = x if fmt == "bf16" else 0x7F + 0x80 * (j & 1)
                    clean_v.view(raw.dtype)[e, o, h, (ch + j) % 128] = 0
            planted.append((b, t, h, bad.numpy()))
    return dict(c, k=k, v=v, ks=ks, vs=vs), dict(c, k=k, v=clean_v, ks=ks, vs=clean_vs), planted


@pytest.mark.parametrize("fmt,scales", [("bf16", None), ("fp8", "head"), ("fp8", "token"), ("int8", "token")])
@pytest.mark.parametrize("nq,hq,hkv,lengths", [
    (17, 4, 4, [517, 17, 129, 300]), (32, 4, 2, [517, 40, 128, 2000]), (150, 2, 2, [517, 150, 385, 256]),
    (64, 24, 8, [3000, 65, 700]), (257, 32, 8, [2900, 257, 400, 700])])
@pytest.mark.parametrize("page", [16, 4])
@pytest.mark.parametrize("bound", [None, 8192])
def test_rows_values_that_are_not_finite_reach_only_the_rows_that_see_them(fmt, scales, nq, hq, hkv, lengths, page, bound):
    """A row gets the infinities and NaN of the tokens it sees, in their channels, and nothing of the others: of later
    queries' tokens, and of stale slots behind a sequence's end. (Weights here are far from underflow.)"""
    from bpt_amd import paged_decode_attention

    c = make_case(fmt, lengths, hq=hq, hkv=hkv, nq=nq, page=page, scales=scales, seed=nq, outliers=False)
    c = c if bound is None else longer_bound(c, bound)
    dirty, clean, planted = plant_nonfinite(c, nq)
    scale = 0.02
    _, want = run_case(clean, scale=scale, out_dtype=torch.float32)
    got = paged_decode_attention(dirty["q"], dirty["k"], dirty["v"], dirty["table"], dirty["lens"], dirty["ks"], dirty["vs"],
                                 scale=scale, max_context=bound or max(lengths), out_dtype=torch.float32).cpu().numpy()
    with np.errstate(invalid="ignore"):
        for b, t, h, bad in planted:
            first = max(t - (lengths[b] - nq), 0)  # the first query that sees token t
            want[b, first:, h * (hq // hkv):(h + 1) * (hq // hkv)] += np.where(np.isfinite(bad), 0, bad)
    fin = np.isfinite(want)
    assert np.array_equal(np.isfinite(got), fin)
    assert np.array_equal(got[~fin], want[~fin], equal_nan=True)
    assert np.abs(got[fin] - want[fin]).max() <= 2.0**-14 * np.abs(want[fin]).max()


@pytest.mark.parametrize("fmt,scales", [("fp8", "token"), ("bf16", None)])
@pytest.mark.parametrize("nq,tile", [(20, 32), (40, 64), (128, 128), (200, 256)])
def test_rows_at_the_longest_tile_line(fmt, scales, nq, tile):
    """2048 sequences of one tile each fill the line in LDS (4096 entries) beside the chunk buffers of every tile size: a
    launch that asked for too much would be refused. The first, some middle and the last sequences against the oracle."""
    from bpt_amd import decode_plan, paged_decode_attention

    g = torch.Generator().manual_seed(nq)
    lengths = torch.randint(0, 2 * nq, (2048,), generator=g).tolist()
    c = make_case(fmt, lengths, hq=1, hkv=1, nq=nq, scales=scales, seed=nq)
    args = (c["q"], c["k"], c["v"], c["table"], c["lens"], c["ks"], c["vs"])
    plan = decode_plan(*args, scale=0.0883883, max_context=512)
    assert plan[1] == 128 and plan[2] == -(-2 * plan[0] * tile * 129 * 4 // 256) * 256
    got = paged_decode_attention(*args, scale=0.0883883, max_context=512)
    for at in (slice(0, 4), slice(1023, 1026), slice(2045, 2048)):
        part = dict(c, q=c["q"][at], table=c["table"][at], lens=c["lens"][at])
        check(got[at], run_case(part)[1], f"{fmt} {nq} queries, sequences {at}")
