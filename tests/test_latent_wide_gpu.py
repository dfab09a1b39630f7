"""Latent attention over entries of 512 + 64 values against float64: head counts around the waves' shares, page and split remainders,
windows, sinks, prefill tiles."""

import pytest
import torch

from vllm_production_stack_amd import ops
from vllm_production_stack_amd.ops import latent

pytestmark = pytest.mark.gpu
DEV, BF = torch.device("cuda"), torch.bfloat16
RANK, ROT, PAGE = 512, 64, 64


def setup(ctx, rows_of, heads, seed):
    g = torch.Generator(device=DEV).manual_seed(seed)
    n = [-(-c // PAGE) for c in ctx]
    pool = (torch.randn(sum(n) + 1, 8 + PAGE * (RANK + ROT), generator=g, device=DEV) * 0.5).to(BF)
    order = torch.randperm(sum(n), generator=g, device=DEV).int().tolist()
    table, at = [], 0
    for k in n:
        table.append(order[at:at + k] + [0] * (max(n) - k))
        at += k
    t = sum(rows_of)
    q = (torch.randn(t, heads, RANK + ROT, generator=g, device=DEV) * 0.7).to(BF)
    return pool, torch.tensor(table, dtype=torch.int32, device=DEV), q, torch.randn(heads, generator=g, device=DEV)


def expected(pool, table, q, sink, ctx, rows_of, scale, window):
    out, at = [], 0
    for s, (c, n) in enumerate(zip(ctx, rows_of)):
        ent = pool[table[s, : -(-c // PAGE)].long(), 8:].reshape(-1, RANK + ROT)[:c].double()
        sc = (q[at:at + n].double().reshape(-1, RANK + ROT) @ ent.t()).view(n, -1, c) * scale
        pos = torch.arange(c - n, c, device=DEV)[:, None, None]
        key = torch.arange(c, device=DEV)[None, None]
        sc.masked_fill_((key > pos) | (key <= pos - window), float("-inf"))
        p = torch.softmax(torch.cat([sc, sink.double().view(1, -1, 1).expand(n, -1, 1)], 2), 2)[..., :c]
        out.append((p.reshape(-1, c) @ ent[:, :RANK]).view(n, -1, RANK))
        at += n
    return torch.cat(out)


@pytest.mark.parametrize("heads", [1, 16, 17, 32, 33, 64, 70])
@pytest.mark.parametrize("splits,window", [(1, 1 << 30), (3, 1 << 30), (8, 100)])
def test_decode_rows(heads, splits, window):
    ctx = [1, 64, 65, 127, 300, 1000]
    pool, table, q, sink = setup(ctx, [1] * len(ctx), heads, heads)
    pos = torch.tensor([c - 1 for c in ctx], dtype=torch.int32, device=DEV)
    out = ops.latent_attention(q[..., :RANK], q[..., RANK:], pool, 8, table, None, pos, sink, 0.05, splits=splits, window=window)
    want = expected(pool, table, q, sink, ctx, [1] * len(ctx), 0.05, window)
    # weights and results in 16 bits: half a unit in the last place each, 2^-9 of the norm
    assert float((out.double() - want).norm() / want.norm()) < 6e-3


@pytest.mark.parametrize("heads,splits", [(16, 1), (32, 1), (32, 4)])
def test_weights_are_not_rounded_to_16_bits(heads, splits):
    ctx = [100, 64, 200, 640, 33]
    pool, table, q, sink = setup(ctx, [1] * len(ctx), heads, 50 + heads)
    pos = torch.tensor([c - 1 for c in ctx], dtype=torch.int32, device=DEV)
    out = ops.latent_attention(q[..., :RANK], q[..., RANK:], pool, 8, table, None, pos, sink, 0.05, splits=splits)
    want = expected(pool, table, q, sink, ctx, [1] * len(ctx), 0.05, 1 << 30)
    # only the result is: an error evenly spread over half a unit in the last place is 2^-9 / sqrt(3) of a power of two, 1.7e-3 of
    # values spread over a binade; weights in 16 bits add as much again
    assert float((out.double() - want).norm() / want.norm()) < 1.8e-3


@pytest.mark.parametrize("heads,rows,splits,window", [(16, 43, 6, 1 << 30), (32, 100, 8, 1 << 30), (64, 33, 8, 1 << 30), (16, 90, 3, 200), (70, 300, 2, 64)])
def test_decode_batches_beyond_a_round(heads, rows, splits, window):
    """More workgroups than CUs: fewer ranges are used than the caller's workspace holds, and some rows see one page or one key."""
    ctx = [1 + (37 * i * i) % 900 for i in range(rows)]
    pool, table, q, sink = setup(ctx, [1] * rows, heads, rows)
    pos = torch.tensor([c - 1 for c in ctx], dtype=torch.int32, device=DEV)
    out = ops.latent_attention(q[..., :RANK], q[..., RANK:], pool, 8, table, None, pos, sink, 0.05, splits=splits, window=window)
    want = expected(pool, table, q, sink, ctx, [1] * rows, 0.05, window)
    assert float((out.double() - want).norm() / want.norm()) < 6e-3   # as above


@pytest.mark.parametrize("heads,rows,bucket", [(16, 36, 40), (32, 33, 40), (32, 65, 80), (16, 100, 128), (70, 20, 24)])
def test_padded_and_unpadded_batches_sum_alike(heads, rows, bucket):
    """The rows of an eager step and of the captured step that holds more rows: equal bits."""
    ctx = [700 + (531 * i) % 3000 for i in range(rows)]
    pool, table, q, sink = setup(ctx, [1] * rows, heads, rows)
    pos = torch.tensor([c - 1 for c in ctx], dtype=torch.int32, device=DEV)
    splits = ops.decode_num_splits(bucket, 1, 32768)
    assert bucket * splits > 256   # more workgroups than CUs: the kernel chooses among the ranges
    pad = torch.nn.functional.pad
    more = bucket - rows
    graph = ops.latent_attention(pad(q, (0, 0, 0, 0, 0, more))[..., :RANK], pad(q, (0, 0, 0, 0, 0, more))[..., RANK:], pool, 8,
                                 pad(table, (0, 0, 0, more)), None, pad(pos, (0, more)), sink, 0.05, splits=splits)
    eager = ops.latent_attention(q[..., :RANK], q[..., RANK:], pool, 8, table, None, pos, sink, 0.05, splits=splits, bucket=bucket)
    assert torch.equal(eager, graph[:rows])


@pytest.mark.parametrize("heads", [3, 16, 64])
def test_prefill_tiles(heads):
    ctx, rows_of = [70, 500, 130], [70, 33, 1]
    pool, table, q, sink = setup(ctx, rows_of, heads, 90 + heads)
    seq = torch.tensor([s for s, n in enumerate(rows_of) for _ in range(n)], dtype=torch.int32, device=DEV)
    pos = torch.cat([torch.arange(c - n, c, dtype=torch.int32) for c, n in zip(ctx, rows_of)]).to(DEV)
    tiles = torch.from_numpy(ops.build_latent_tiles(rows_of, ctx, heads)).to(DEV)
    out = ops.latent_attention(q[..., :RANK], q[..., RANK:], pool, 8, table, seq, pos, sink, 0.05, tiles=tiles)
    want = expected(pool, table, q, sink, ctx, rows_of, 0.05, 1 << 30)
    assert float((out.double() - want).norm() / want.norm()) < 6e-3


@pytest.mark.parametrize("heads,rows_of,ctx,window", [
    (16, [20], [3000], 1 << 30), (32, [3, 40], [200, 1500], 1 << 30), (64, [70], [1100], 1 << 30), (16, [9, 1, 130], [9, 513, 700], 1 << 30),
    (32, [50], [2000], 300), (7, [33], [640], 1 << 30), (32, [50], [2000], 900), (16, [30, 7], [3000, 60], 1500)])
def test_prefill_tiles_cut_along_the_keys(heads, rows_of, ctx, window, monkeypatch):
    """Lists of few tiles: ranges of the keys and a merge, tiles that see fewer pages than the list has ranges, an unused entry."""
    pool, table, q, sink = setup(ctx, rows_of, heads, 7 + heads)
    table = torch.nn.functional.pad(table, (0, 60))   # wider than the longest context
    tiles = torch.from_numpy(ops.build_latent_tiles(rows_of, ctx, heads)).to(DEV)
    tiles = torch.cat([tiles, torch.full((1, 6), -1, dtype=torch.int32, device=DEV)])
    assert latent.latent_tile_splits(tiles.shape[0], table.shape[1], RANK, ROT, True) > 1
    seq = torch.tensor([i for i, n in enumerate(rows_of) for _ in range(n)], dtype=torch.int32, device=DEV)
    pos = torch.tensor([c - n + k for n, c in zip(rows_of, ctx) for k in range(n)], dtype=torch.int32, device=DEV)
    asked, cut = [], latent.latent_tile_splits
    monkeypatch.setattr(latent, "latent_tile_splits", lambda *a: asked.append(a) or cut(*a))
    out = ops.latent_attention(q[..., :RANK], q[..., RANK:], pool, 8, table, seq, pos, sink, 0.05, tiles=tiles, window=window)
    want = expected(pool, table, q, sink, ctx, rows_of, 0.05, window)
    assert float((out.double() - want).norm() / want.norm()) < 6e-3   # as above
    assert asked == [(tiles.shape[0], table.shape[1], RANK, ROT, True, window)]
