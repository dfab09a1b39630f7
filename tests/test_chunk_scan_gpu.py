"""The block form of the recurrences (``csrc/kernels/chunk_scan.hip``) against the float64 recurrence where `test_retention_gpu.py` does
not reach: gates per channel, gates whose products leave the range of 32 bits, whole sequences without pieces, several states at once."""

import pytest
import torch

from vllm_production_stack_amd import ops
from vllm_production_stack_amd.ops import seqmix

pytestmark = pytest.mark.gpu
DEV = torch.device("cuda")


def i32(x):
    return torch.tensor(x, dtype=torch.int32, device=DEV)


def gated(heads, vdim, lens, starts, lower, bias, seed=0, slots=None, pieces=True, resets=()):
    """(outputs, expected, states, expected states) of one call; ``lower`` / ``bias``: (least, most) per channel; ``resets``: rows
    whose gates are nothing in every fifth channel."""
    g = torch.Generator().manual_seed(seed)
    t, hd = sum(lens), heads * 128
    proj = torch.randn(t, 2 * hd + heads * vdim, generator=g).bfloat16()
    lo = torch.rand(hd, generator=g) * (lower[1] - lower[0]) + lower[0]
    b = torch.rand(hd, generator=g) * (bias[1] - bias[0]) + bias[0]
    if resets:
        lo[::5] = 0
        proj[list(resets), hd:2 * hd] = -60
    slots = list(range(len(lens))) if slots is None else slots
    state = torch.randn(len(lens), hd * vdim + 4, generator=g)
    pj = proj.double()
    q, z, v = (pj[:, o:o + heads * n].view(t, heads, n) for o, n in ((0, 128), (hd, 128), (2 * hd, vdim)))
    a = lo.double().view(heads, 128) + (1 - lo.double().view(heads, 128)) * torch.sigmoid(z + b.double().view(heads, 128))
    q = torch.nn.functional.silu(q)
    want, ends, row = [], state.double()[:, 4:].clone(), 0
    for s, n in enumerate(lens):
        S = ends[slots[s]].view(heads, 128, vdim).clone() if slots[s] >= 0 else torch.zeros(heads, 128, vdim, dtype=torch.float64)
        S = S * (0 if starts[s] == 0 else 1)
        for i in range(row, row + n):
            S = S * a[i, :, :, None] + (1 - a[i])[:, :, None] * v[i, :, None, :]
            want.append((S * q[i, :, :, None]).sum(1) * (1 if slots[s] >= 0 else 0))
        if slots[s] >= 0:
            ends[slots[s]] = S.reshape(-1)
        row += n
    cu = [sum(lens[:i]) for i in range(len(lens) + 1)]
    pos = torch.cat([torch.arange(p, p + n) for p, n in zip(starts, lens)]).int().to(DEV)
    cut = ops.build_scan_pieces(lens, target=6) if pieces else None
    st = state.to(DEV)
    out = ops.recurrent_scan(proj.to(DEV), 0, hd, 2 * hd, heads, 128, vdim, st, 4, i32(cu), i32(slots), pos, gate_bias=b.to(DEV),
                             gate_lower=lo.to(DEV), pieces=None if cut is None else tuple(torch.from_numpy(c).to(DEV) for c in cut))
    return out, torch.stack(want), st[:, 4:], ends


def off(got, want):
    return float((got.double().cpu() - want).norm() / want.norm())


# remainders of blocks, runs of several pieces, continued and fresh sequences; steps without pieces go whole
@pytest.mark.parametrize("heads,vdim,lens,starts,pieces", [
    (2, 128, [300], [0], True), (1, 256, [33, 290], [5, 0], True), (3, 128, [31, 257, 1], [0, 64, 9], True),
    (2, 128, [32], [3], False), (2, 256, [65, 2, 130], [0, 1, 7], False), (1, 128, [256], [0], True)])
def test_gated_blocks(heads, vdim, lens, starts, pieces):
    out, want, st, ends = gated(heads, vdim, lens, starts, (0.2, 0.9), (1.0, 3.0), pieces=pieces)
    # sums of 128 channels in 32 bits and gates one rounding off: a few units in the last place
    assert off(out, want) < 5e-7 and off(st, ends) < 1e-6


# a block's product of gates below 2^-60: mean logits from -3 to -40 (gates of 0.05 down to exactly 0) take shorter blocks
@pytest.mark.parametrize("bias", [(-4.0, -2.0), (-12.0, 2.0), (-130.0, 3.0)])
def test_gates_that_forget_at_once(bias):
    for lens, pieces in (([300], True), ([90], False)):
        out, want, st, ends = gated(2, 128, lens, [4] * len(lens), (0.0, 0.0), bias, seed=3, pieces=pieces)
        assert off(out, want) < 5e-7 and off(st, ends) < 1e-6


# gates that are nothing now and then among others that last: blocks that shrink and grow again, runs that end token by token, runs that
# begin or end with such a token, sequences too short for a second try
@pytest.mark.parametrize("vdim", [128, 256])
@pytest.mark.parametrize("lens,pieces,every,first", [([700], True, 7, 3), ([700], True, 45, 0), ([900, 300], True, 250, 31), ([300], False, 100, 50),
                                                     ([20, 9, 40], False, 20, 5), ([33], False, 33, 32), ([130], False, 16, 15)])
def test_gates_that_forget_now_and_then(vdim, lens, pieces, every, first):
    resets = range(first, sum(lens), every)
    out, want, st, ends = gated(2, vdim, lens, [4] * len(lens), (0.2, 0.9), (1.0, 3.0), seed=7, pieces=pieces, resets=resets)
    assert off(out, want) < 5e-7 and off(st, ends) < 1e-6


@pytest.mark.parametrize("bias", [(-4.0, -2.0), (-12.0, 2.0), (-130.0, 3.0)])
def test_token_by_token_rounds_no_more_than_one_value(bias):
    """Runs that go token by token: gates, keys and queries in 32 bits with about one rounding each, a channel's part of an output in
    chains of 16: together below the largest rounding of one value, 2^-24 (5.2e-8; one chain of 32 and quotients of rounded sums 6.3e-8)."""
    out, want, st, ends = gated(2, 128, [300, 33], [4, 4], (0.0, 0.0), bias, seed=3)
    assert off(out, want) < 2 ** -24 and off(st, ends) < 2 ** -24


def test_gates_that_forget_cost_a_few_times_the_others():
    """Token by token a run takes about three times as long as in blocks of 32 tokens; in blocks that shrink to one token it took 27."""
    heads, t = 32, 4096
    hd = heads * 128
    g = torch.Generator(device=DEV).manual_seed(2)
    proj = torch.randn(t, 3 * hd, generator=g, device=DEV).bfloat16()
    state, lower = torch.zeros(1, hd * 128, device=DEV), torch.zeros(hd, device=DEV)
    pieces = tuple(torch.from_numpy(c).to(DEV) for c in ops.build_scan_pieces([t]))
    pos, cu, slot = torch.arange(t, dtype=torch.int32, device=DEV), i32([0, t]), i32([0])

    def time(logit):
        bias, best = torch.full((hd,), logit, device=DEV), float("inf")
        for _ in range(6):
            a, b = torch.cuda.Event(enable_timing=True), torch.cuda.Event(enable_timing=True)
            a.record()
            ops.recurrent_scan(proj, 0, hd, 2 * hd, heads, 128, 128, state, 0, cu, slot, pos, gate_bias=bias, gate_lower=lower, pieces=pieces)
            b.record()
            b.synchronize()
            best = min(best, a.elapsed_time(b))
        return best

    usual = time(2.0)
    assert max(time(logit) for logit in (-6.0, -14.0, -40.0)) < 6 * usual


def test_rows_of_no_sequence():
    out, want, st, ends = gated(2, 128, [40, 60], [0, 8], (0.2, 0.9), (1.0, 3.0), slots=[-1, 1], pieces=False)
    assert (out[:40] == 0).all() and off(out, want) < 5e-7 and off(st, ends) < 1e-6


@pytest.mark.parametrize("t,pieces", [(70, False), (300, True)])
def test_a_value_that_is_not_finite_stays_in_its_column(t, pieces):
    g = torch.Generator().manual_seed(5)
    hd = 128
    cut = ops.build_scan_pieces([t], target=6) if pieces else None
    cut = None if cut is None else tuple(torch.from_numpy(c).to(DEV) for c in cut)
    proj = torch.randn(t, 3 * hd, generator=g).bfloat16().to(DEV)
    proj[40, 2 * hd + 7] = float("inf")
    args = (i32([0, t]), i32([0]), torch.arange(t, dtype=torch.int32, device=DEV))
    out = ops.recurrent_scan(proj, 0, hd, 2 * hd, 1, 128, 128, torch.zeros(1, 128 * 128, device=DEV), 0, *args,
                             gate_bias=torch.ones(128, device=DEV), gate_lower=torch.full((128,), 0.5, device=DEV), pieces=cut)
    bad = ~torch.isfinite(out[:, 0])
    assert bad[40:, 7].all() and int(bad.sum()) == t - 40
    # and it stays as it was beside a step in which the value is finite
    proj[40, 2 * hd + 7] = 1.0
    ref = ops.recurrent_scan(proj, 0, hd, 2 * hd, 1, 128, 128, torch.zeros(1, 128 * 128, device=DEV), 0, *args,
                             gate_bias=torch.ones(128, device=DEV), gate_lower=torch.full((128,), 0.5, device=DEV), pieces=cut)
    keep = [i for i in range(128) if i != 7]
    assert off(out[:, 0, keep], ref[:, 0, keep].double().cpu()) < 5e-7


@pytest.mark.parametrize("vdim,act", [(256, True), (128, False)])
def test_fixed_decay_without_pieces_matches_the_walk(vdim, act):
    """Sequences of 8 rows and more on average go in blocks; the same rows in calls of single sequences below that go token by token."""
    g = torch.Generator().manual_seed(1)
    heads, lens = 2, [40, 9, 33]
    hd = heads * 128
    proj = torch.randn(sum(lens), 2 * hd + heads * vdim, generator=g).bfloat16().to(DEV)
    decay = torch.tensor([0.97, 0.4], device=DEV)
    start = torch.randn(3, heads * 128 * vdim, generator=g).to(DEV)
    pos = torch.cat([torch.arange(3, 3 + n) for n in lens]).int().to(DEV)
    cols = (0, hd, 2 * hd, heads, 128, vdim)
    whole = start.clone()
    out = ops.recurrent_scan(proj, *cols, whole, 0, i32([0, 40, 49, 82]), i32([0, 1, 2]), pos, decay=decay, act=act, min_decay=0.4)
    step, rows, at = start.clone(), [], 0
    for s, n in enumerate(lens):
        for k in range(0, n, seqmix.SCAN_BLOCK_MIN_ROWS - 1):
            m = min(seqmix.SCAN_BLOCK_MIN_ROWS - 1, n - k)
            rows.append(ops.recurrent_scan(proj[at:at + m], *cols, step, 0, i32([0, m]), i32([s]), pos[at:at + m], decay=decay, act=act))
            at += m
    assert off(out, torch.cat(rows).double().cpu()) < 5e-7 and off(whole, step.double().cpu()) < 5e-7
