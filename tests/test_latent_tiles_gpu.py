"""Tiles of 64 (token, head) pairs over latent entries against float64: fillings around the waves' and fragments' sixteen slots, ends of
pages, windows, rows of more than 32 heads, cut lists, queries and results in larger tensors, scores that differ by many powers of two."""

import pytest
import torch

from test_latent_wide_gpu import BF, DEV, RANK, expected, setup
from vllm_production_stack_amd import ops

pytestmark = pytest.mark.gpu


def close(got, pool, table, q, sink, ctx, rows_of, scale, window=1 << 30):
    """Weights and result in 16 bits, eight of them significand: 2^-8 of each weight, so of the sum of absolute values, and of the result."""
    want = expected(pool, table, q, sink, ctx, rows_of, scale, window)
    size = pool.clone()
    size[:, 8:] = size[:, 8:].abs()
    weights = expected_of_sizes(pool, size, table, q, sink, ctx, rows_of, scale, window)
    err = (got.double() - want).abs()
    assert bool((err <= 2 ** -8 * want.abs() + 1.05 * 2 ** -8 * weights + 1e-5).all()), float(err.max())


def expected_of_sizes(pool, size, table, q, sink, ctx, rows_of, scale, window):
    """The sums with the values' absolute values: entries whose value part is |v| and whose scores are those of v."""
    out, at = [], 0
    for s, (c, n) in enumerate(zip(ctx, rows_of)):
        pages = table[s, : -(-c // 64)].long()
        ent, mag = (x[pages, 8:].reshape(-1, 576)[:c].double() for x in (pool, size))
        sc = (q[at:at + n].double().reshape(-1, 576) @ ent.t()).view(n, -1, c) * scale
        pos, key = torch.arange(c - n, c, device=DEV)[:, None, None], torch.arange(c, device=DEV)[None, None]
        sc.masked_fill_((key > pos) | (key <= pos - window), float("-inf"))
        p = torch.softmax(torch.cat([sc, sink.double().view(1, -1, 1).expand(n, -1, 1)], 2), 2)[..., :c]
        out.append((p.reshape(-1, c) @ mag[:, :RANK]).view(n, -1, RANK))
        at += n
    return torch.cat(out)


@pytest.mark.parametrize("heads,rows_of,ctx,window", [
    (1, [1, 64, 65], [1, 64, 200], 1 << 30), (5, [13, 1], [77, 129], 1 << 30), (15, [5, 4], [5, 400], 1 << 30), (16, [17], [145], 30),
    (33, [3], [64], 1 << 30), (48, [2, 2], [63, 192], 64), (64, [3], [1030], 1 << 30), (100, [3, 1], [66, 257], 1 << 30),
    (32, [2], [2000], 1 << 30), (16, [8], [1500], 700)])
@pytest.mark.parametrize("scale", [0.05, 0.7])
def test_fillings_of_a_tile(heads, rows_of, ctx, window, scale):
    pool, table, q, sink = setup(ctx, rows_of, heads, 3 * heads + len(ctx))
    wide = torch.randn(q.shape[0], heads + 1, 640, device=DEV).to(BF)   # queries with others between them
    wide[:, 1:, :576] = q
    lat, rot = wide[:, 1:, :512], wide[:, 1:, 512:576]
    seq = torch.tensor([s for s, n in enumerate(rows_of) for _ in range(n)], dtype=torch.int32, device=DEV)
    pos = torch.cat([torch.arange(c - n, c, dtype=torch.int32) for c, n in zip(ctx, rows_of)]).to(DEV)
    tiles = torch.from_numpy(ops.build_latent_tiles(rows_of, ctx, heads)).to(DEV)
    buf = torch.full((q.shape[0], heads + 1, RANK + 8), 7.0, dtype=BF, device=DEV)
    ops.latent_attention(lat, rot, pool, 8, table, seq, pos, sink, scale, out=buf[:, :heads, :RANK], tiles=tiles, window=window)
    close(buf[:, :heads, :RANK], pool, table, q, sink, ctx, rows_of, scale, window)
    assert bool((buf[:, heads] == 7).all()) and bool((buf[..., RANK:] == 7).all())


@pytest.mark.parametrize("heads,splits,window", [(33, 1, 1 << 30), (64, 5, 1 << 30), (70, 2, 130), (128, 1, 64)])
def test_rows_of_more_than_32_heads(heads, splits, window):
    ctx = [1, 63, 64, 65, 128, 129, 700]
    pool, table, q, sink = setup(ctx, [1] * len(ctx), heads, heads)
    pos = torch.tensor([c - 1 for c in ctx], dtype=torch.int32, device=DEV)
    got = ops.latent_attention(q[..., :RANK], q[..., RANK:], pool, 8, table, None, pos, sink, 0.3, splits=splits, window=window)
    close(got, pool, table, q, sink, ctx, [1] * len(ctx), 0.3, window)


def test_no_sink_a_sink_of_no_weight_and_a_nan():
    pool, table, q, _ = setup([90, 90], [20, 20], 16, 5)
    seq = torch.tensor([0] * 20 + [1] * 20, dtype=torch.int32, device=DEV)
    pos = torch.arange(70, 90, dtype=torch.int32, device=DEV).repeat(2)
    tiles = torch.from_numpy(ops.build_latent_tiles([20, 20], [90, 90], 16)).to(DEV)
    none = torch.full((16,), float("-inf"), device=DEV)
    got = [ops.latent_attention(q[..., :RANK], q[..., RANK:], pool, 8, table, seq, pos, s, 0.3, tiles=tiles) for s in (None, none)]
    assert torch.equal(*got)
    close(got[0], pool, table, q, none, [90, 90], [20, 20], 0.3)
    q2 = q.clone()
    q2[3, 2, 5] = float("nan")  # one (token, head) pair: nothing else changes
    got2 = ops.latent_attention(q2[..., :RANK], q2[..., RANK:], pool, 8, table, seq, pos, None, 0.3, tiles=tiles)
    assert bool(got2[3, 2].isnan().all())
    got2[3, 2] = got[0][3, 2]
    assert torch.equal(got2, got[0])


@pytest.mark.parametrize("scale", [-0.3, 0.0, 1e-42])
def test_scales_of_any_sign(scale):
    """Scores turn their order with a negative scale and mean nothing with one of zero; a window that some pages' slots see nothing of."""
    rows_of, ctx, heads = [40, 5], [300, 5], 16
    pool, table, q, sink = setup(ctx, rows_of, heads, 11)
    seq = torch.tensor([0] * 40 + [1] * 5, dtype=torch.int32, device=DEV)
    pos = torch.cat([torch.arange(c - n, c, dtype=torch.int32) for c, n in zip(ctx, rows_of)]).to(DEV)
    tiles = torch.from_numpy(ops.build_latent_tiles(rows_of, ctx, heads)).to(DEV)
    for window in (1 << 30, 66):
        got = ops.latent_attention(q[..., :RANK], q[..., RANK:], pool, 8, table, seq, pos, sink, scale, tiles=tiles, window=window)
        close(got, pool, table, q, sink, ctx, rows_of, scale, window)


@pytest.mark.parametrize("scale", [-0.3, 0.0, 1e-42])
@pytest.mark.parametrize("heads,splits", [(16, 1), (32, 3)])
def test_decode_rows_with_scales_of_any_sign(scale, heads, splits):
    ctx = [1, 64, 65, 500]
    pool, table, q, sink = setup(ctx, [1] * len(ctx), heads, heads)
    pos = torch.tensor([c - 1 for c in ctx], dtype=torch.int32, device=DEV)
    for window in (1 << 30, 70):
        got = ops.latent_attention(q[..., :RANK], q[..., RANK:], pool, 8, table, None, pos, sink, scale, splits=splits, window=window)
        close(got, pool, table, q, sink, ctx, [1] * len(ctx), scale, window)


@pytest.mark.parametrize("tiled", [True, False])
@pytest.mark.parametrize("heads", [16, 40])
def test_a_sink_or_scale_that_is_no_number_reaches_the_result(tiled, heads):
    ctx, rows_of = ([90], [20]) if tiled else ([90, 7], [1, 1])
    pool, table, q, sink = setup(ctx, rows_of, heads, 3)
    seq = torch.zeros(20, dtype=torch.int32, device=DEV) if tiled else None
    pos = torch.cat([torch.arange(c - n, c, dtype=torch.int32) for c, n in zip(ctx, rows_of)]).to(DEV)
    kw = {"tiles": torch.from_numpy(ops.build_latent_tiles(rows_of, ctx, heads)).to(DEV)} if tiled else {"splits": 1}
    run = lambda s, scale: ops.latent_attention(q[..., :RANK], q[..., RANK:], pool, 8, table, seq, pos, s, scale, **kw)
    want, nan = run(sink, 0.3), sink.clone()
    nan[3] = float("nan")  # one head: nothing else changes
    got = run(nan, 0.3)
    assert bool(got[:, 3].isnan().all())
    got[:, 3] = want[:, 3]
    assert torch.equal(got, want)
    assert bool(run(sink, float("nan")).isnan().all())


@pytest.mark.parametrize("tiled", [True, False])
@pytest.mark.parametrize("heads", [16, 40])
def test_what_is_no_number_reaches_the_result_over_key_ranges(tiled, heads):
    """The same where several ranges hold a row and a merge joins them, and an infinite sink, which leaves the entries no weight."""
    ctx, rows_of = ([1500], [20]) if tiled else ([1500, 7, 300], [1, 1, 1])
    pool, table, q, sink = setup(ctx, rows_of, heads, 3)
    seq = torch.zeros(20, dtype=torch.int32, device=DEV) if tiled else None
    pos = torch.cat([torch.arange(c - n, c, dtype=torch.int32) for c, n in zip(ctx, rows_of)]).to(DEV)
    kw = {"splits": 3}
    if tiled:
        kw = {"tiles": torch.from_numpy(ops.build_latent_tiles(rows_of, ctx, heads)).to(DEV)}
        assert ops.latent.latent_tile_splits(kw["tiles"].shape[0], table.shape[1], RANK, 64, True) > 1
    run = lambda s, scale=0.3, q=q: ops.latent_attention(q[..., :RANK], q[..., RANK:], pool, 8, table, seq, pos, s, scale, **kw)
    nan, inf, q2 = sink.clone(), sink.clone(), q.clone()
    nan[3], inf[3], q2[1, 2, 5] = float("nan"), float("inf"), float("nan")
    for s in (sink, None):
        want = run(s)
        assert bool(want.isfinite().all())
        got = run(s, q=q2)  # one (token, head) pair: nothing else changes
        assert bool(got[1, 2].isnan().all())
        got[1, 2] = want[1, 2]
        assert torch.equal(got, want)
        assert bool(run(s, float("nan")).isnan().all())
    want, got, none = run(sink), run(nan), run(inf)
    assert bool(got[:, 3].isnan().all()) and bool((none[:, 3] == 0).all())
    got[:, 3] = none[:, 3] = want[:, 3]
    assert torch.equal(got, want) and torch.equal(none, want)
