"""The block form of the fixed-decay recurrence against the float64 recurrence: block and run remainders, both rotations and
partial ones, silu inputs, continued and fresh sequences, rows of no sequence, values that are not finite."""

import pytest
import torch

import revelix_oracle as ro
from vllm_production_stack_amd import ops
from vllm_production_stack_amd.ops import seqmix

pytestmark = pytest.mark.gpu
DEV = torch.device("cuda")


def i32(x):
    return torch.tensor(x, dtype=torch.int32, device=DEV)


def inputs(heads, vdim, lens, starts, decay, rot, layout, act, seed=0):
    """(call, expected outputs, expected states): state slots hold something for sequences that continue."""
    g = torch.Generator().manual_seed(seed)
    t, dim = sum(lens), 128
    width = 8 + heads * (2 * dim + vdim)
    proj = torch.randn(t, width, generator=g).bfloat16()
    cols = (8, 8 + heads * dim, 8 + 2 * heads * dim)
    table = ops.build_cos_sin(rot, 4096, 777.0) if rot else None
    state = torch.randn(len(lens), heads * dim * vdim + 4, generator=g)
    pos = torch.cat([torch.arange(p, p + n) for p, n in zip(starts, lens)])
    pj = proj.double()
    q, k, v = (pj[:, c:c + heads * d].view(t, heads, d) for c, d in zip(cols, (dim, dim, vdim)))
    if act:
        q, k, v = (torch.nn.functional.silu(x) for x in (q, k, v))
    if rot:  # the table's own 32-bit cosines: what is tested is the recurrence
        r = {"base": 777.0, "dims": rot}
        q, k = (ro.rotate(x, pos, r, "half" if layout == 0 else "pairs") for x in (q, k))
    k = k * 0.25
    want, ends, row = [], [], 0
    d = torch.tensor(decay, dtype=torch.float32).double().view(heads, 1, 1)
    for s, n in enumerate(lens):
        S = state[s, 4:].double().view(heads, dim, vdim) * (0 if starts[s] == 0 else 1)
        for i in range(row, row + n):
            S = S * d + k[i, :, :, None] * v[i, :, None, :]
            want.append((S * q[i, :, :, None]).sum(1))
        ends.append(S.reshape(-1))
        row += n
    cut = ops.build_scan_pieces(lens, target=6)
    kw = dict(decay=torch.tensor(decay, device=DEV), cos_sin=None if table is None else table.to(DEV), rot_dims=rot, layout=layout,
              k_scale=0.25, act=act, pieces=tuple(torch.from_numpy(c).to(DEV) for c in cut))
    cu = [0]
    for n in lens:
        cu.append(cu[-1] + n)
    call = [proj.to(DEV), *cols, heads, dim, vdim, state.to(DEV), 4, i32(cu), i32(list(range(len(lens)))), pos.int().to(DEV)]
    return call, kw, torch.stack(want), torch.stack(ends)


def off(got, want):
    return float((got.double().cpu() - want).norm() / want.norm())


SHAPES = [
    (2, 256, [128], [0], 128, 0, False),            # whole blocks, one sequence
    (1, 128, [129, 1, 16, 17], [0, 5, 0, 9], 128, 1, False),   # one token past a block, one-token and half-block sequences
    (3, 256, [150, 333], [40, 0], 64, 0, False),    # partial rotation, a continued sequence first
    (2, 128, [287], [0], 0, 0, True),               # silu inputs
    (2, 256, [160], [7], 8, 1, False),
]


@pytest.mark.parametrize("heads,vdim,lens,starts,rot,layout,act", SHAPES)
def test_blocks_match_the_recurrence(heads, vdim, lens, starts, rot, layout, act):
    decay = [0.999, 0.5, 0.05][:heads]  # the last one's 32nd power is far below what 32 bits can divide by
    call, kw, want, ends = inputs(heads, vdim, lens, starts, decay, rot, layout, act)
    assert seqmix._retention_blocks(call[0], *call[1:4], 128, vdim, kw["cos_sin"], rot, layout)
    out = ops.recurrent_scan(*call, **kw)
    # 32-bit sums over at most 128 channels and a few hundred tokens: a few units in the last place of the norm; the rotation's
    # angles are 32-bit products of positions below 512, off by up to 3e-5 of a turn's derivative in rare channels
    tol = 2e-5 if rot else 2e-6
    assert off(out, want) < tol and off(call[7][:, 4:], ends) < tol


# the smallest decay as the host knows it: a whole block's products in range (just so in the last), which is what the other form needs
@pytest.mark.parametrize("heads,vdim,lens,starts,rot,layout,act", SHAPES)
def test_blocks_of_known_decays(heads, vdim, lens, starts, rot, layout, act):
    for decay in ([0.999, 0.5, 0.9][:heads], [seqmix.SCAN_BLOCK_MIN_DECAY * 1.0001] * heads):
        call, kw, want, ends = inputs(heads, vdim, lens, starts, decay, rot, layout, act)
        out = ops.recurrent_scan(*call, **kw, min_decay=min(decay))
        tol = 2e-5 if rot else 2e-6  # as above
        assert off(out, want) < tol and off(call[7][:, 4:], ends) < tol


def test_decays_that_forget_cost_no_more():
    """Decays that a block's 32 tokens cannot divide by, known or not: as long as others, at most twice the blocks that divide (in
    blocks as short as they would need, 4 to 25 times)."""
    heads, t, vdim = 32, 4096, 128
    g = torch.Generator(device=DEV).manual_seed(2)
    proj = torch.randn(t, heads * (256 + vdim), generator=g, device=DEV).bfloat16()
    state, pos = torch.zeros(1, heads * 128 * vdim, device=DEV), torch.arange(t, dtype=torch.int32, device=DEV)
    pieces = tuple(torch.from_numpy(c).to(DEV) for c in ops.build_scan_pieces([t]))
    args = (proj, 0, heads * 128, heads * 256, heads, 128, vdim, state, 0, i32([0, t]), i32([0]), pos)

    def time(decay, known):
        d, best = torch.full((heads,), decay, device=DEV), float("inf")
        for _ in range(6):
            a, b = torch.cuda.Event(enable_timing=True), torch.cuda.Event(enable_timing=True)
            a.record()
            ops.recurrent_scan(*args, decay=d, pieces=pieces, min_decay=known)
            b.record()
            b.synchronize()
            best = min(best, a.elapsed_time(b))
        return best

    usual = time(0.97, 0.97)
    assert max(time(d, known) for d in (1e-3, 1e-6, 1e-19) for known in (0.0, d)) < 2.5 * usual


@pytest.mark.parametrize("known", [0.0, 0.9])
def test_rows_of_no_sequence_and_values_that_are_not_finite(known):
    call, kw, want, _ = inputs(2, 128, [140, 40], [0, 0], [0.9, 0.99], 0, 0, False, seed=3)
    call[10] = i32([-1, 1])
    call[0][150, call[3]:call[3] + 4] = float("inf")   # token 10 of the second sequence
    before = call[7].clone()
    out = ops.recurrent_scan(*call, **kw, min_decay=known)
    assert (out[:140] == 0).all() and torch.equal(call[7][0], before[0])
    assert off(out[140:150], want[140:150]) < 2e-6     # tokens before it see nothing of it
    assert torch.isfinite(out[140:, 1]).all() and off(out[140:, 1], want[140:, 1]) < 2e-6
    assert not torch.isfinite(out[150:, 0, :4]).any()
    assert torch.isfinite(out[140:, 0, 4:]).all()
