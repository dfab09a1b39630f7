"""Short steps with prompt rows: projection, rotation and cache write in one reduction, against the passes one by one."""

import pytest
import torch

from vllm_production_stack_amd import ops
from vllm_production_stack_amd.models.batch import BatchMeta

DEV = torch.device("cuda")
PAGE, D = 64, 128


def _meta(lens, cached, decode, pad, nq, nkv, split):
    """Decode rows behind 70 tokens, then prompts of ``lens`` rows behind ``cached`` tokens, then ``pad`` rows of no sequence."""
    width = -(-(cached + max(lens)) // PAGE)
    seqs = decode + len(lens)
    table = torch.arange(seqs * width, dtype=torch.int32).flip(0).view(seqs, width)
    at = [(s, 70) for s in range(decode)] + [(decode + i, cached + t) for i, n in enumerate(lens) for t in range(n)]
    slots = [int(table[s, p // PAGE]) * PAGE + p % PAGE for s, p in at] + [-1] * pad
    m = BatchMeta(positions=torch.tensor([p for _, p in at] + [0] * pad, dtype=torch.int32, device=DEV),
                  slots=torch.tensor(slots, dtype=torch.int64, device=DEV), num_decode=decode, num_prefill_seqs=len(lens), pre_padded=pad > 0)
    table = table.to(DEV)
    m.dec_block_tables, m.dec_ctx_lens = table[:decode].contiguous(), torch.full((decode,), 71, dtype=torch.int32, device=DEV)
    ctx = [cached + n for n in lens]
    cu = [0]
    for n in lens:
        cu.append(cu[-1] + n)
    m.pre_block_tables = table[decode:].contiguous()
    m.pre_ctx_lens, m.pre_cu_q = (torch.tensor(v, dtype=torch.int32, device=DEV) for v in (ctx, cu))
    m.pre_tile_rows = ops.prefill_tile_rows(lens, nq, nkv)
    ts, tq = ops.build_prefill_tiles(lens, nq, nkv, m.pre_tile_rows, ctx)
    cut = ops.plan_prefill_splits(ts, tq, lens, ctx, nq, nkv, m.pre_tile_rows)
    assert (cut is not None) == split
    if split:
        ts, tq, spl, groups, records = cut
        m.pre_split, m.pre_split_groups = (torch.tensor(v, dtype=torch.int32, device=DEV) for v in (spl, groups))
        m.pre_split_ws = torch.empty(records * ops.prefill_split_record_bytes(nq, nkv) // 4, dtype=torch.float32, device=DEV)
    m.pre_tile_seq, m.pre_tile_q0 = (torch.tensor(v, dtype=torch.int32, device=DEV) for v in (ts, tq))
    return m, seqs * width


@pytest.mark.gpu
@pytest.mark.parametrize("lens,cached,decode,pad,split", [
    ([1], 0, 0, 0, False), ([17], 300, 0, 0, False), ([40], 400, 3, 0, False), ([64], 1100, 0, 3, True), ([90, 6], 1200, 0, 0, True), ([97], 2100, 0, 0, True),
    ([200, 13], 1200, 2, 5, True), ([256], 1300, 0, 0, True)])
@pytest.mark.parametrize("bias", [False, True])
def test_prompt_attention_block_is_the_passes_one_by_one(lens, cached, decode, pad, split, bias):
    nq, nkv, k = 32, 8, 4096
    g = torch.Generator(device=DEV).manual_seed(7)
    meta, pages = _meta(lens, cached, decode, pad, nq, nkv, split)
    rows = decode + sum(lens) + pad
    x = torch.randn(rows, k, device=DEV, generator=g).bfloat16()
    w = (torch.randn((nq + 2 * nkv) * D, k, device=DEV, generator=g) * 0.02).bfloat16()
    b = torch.randn(w.shape[0], device=DEV, generator=g).bfloat16() if bias else None
    cos_sin = ops.build_cos_sin(D, 4096, 10000.0, device=DEV)
    old = torch.randn(pages, 2, 2, nkv, PAGE * D, device=DEV, generator=g).bfloat16()
    got_pool, want_pool = old.clone(), old.clone()
    got = ops.prompt_attention_block(x, w, b, got_pool, 1, meta, nq, nkv, D, D ** -0.5, cos_sin)
    assert got is not None
    want = ops.attention_block(torch.nn.functional.linear(x, w, b), want_pool, 1, meta, nq, nkv, D, D ** -0.5, cos_sin)
    # sums in another order flip last places of 16 bits, before and after the rotation and in the attention's rows
    assert float((got_pool.float() - want_pool.float()).norm() / (want_pool.float() - old.float()).norm()) < 2 ** -8
    assert torch.equal(got_pool[:, 0], old[:, 0])
    changed = lambda p: (p[:, 1] != old[:, 1]).sum()  # noqa: E731
    assert abs(int(changed(got_pool)) - int(changed(want_pool))) < 0.01 * int(changed(want_pool))
    real = rows - pad
    assert float((got[:real].float() - want[:real].float()).norm() / want[:real].float().norm()) < 1e-2
    if pad:
        assert not got[real:].any()


@pytest.mark.gpu
def test_what_is_not_taken():
    nq, nkv, k = 32, 8, 4096
    meta, pages = _meta([257], 0, 0, 0, nq, nkv, False)
    w = torch.zeros((nq + 2 * nkv) * D, k, device=DEV, dtype=torch.bfloat16)
    pool = torch.zeros(pages, 1, 2, nkv, PAGE * D, device=DEV, dtype=torch.bfloat16)
    cos_sin = ops.build_cos_sin(D, 512, 10000.0, device=DEV)
    args = (w, None, pool, 0, meta, nq, nkv, D, 1.0, cos_sin)
    assert ops.prompt_attention_block(torch.zeros(257, k, device=DEV, dtype=torch.bfloat16), *args) is None  # two row tiles
    x = torch.zeros(64, k, device=DEV, dtype=torch.bfloat16, requires_grad=True)
    assert ops.prompt_attention_block(x, *args) is None  # something follows it
    with torch.no_grad():
        meta.slots = None
        assert ops.prompt_attention_block(x, *args) is None
