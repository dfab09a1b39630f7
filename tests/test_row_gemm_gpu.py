"""Products of a few rows that are whole in one launch: sums of all sizes of tiles, chunks and rows against 64 bits, and a decoder's steps with
and without them."""

import dataclasses

import pytest
import torch

from vllm_production_stack_amd import ops
from vllm_production_stack_amd.engine.config import PRESETS
from vllm_production_stack_amd.models.batch import BatchMeta
from vllm_production_stack_amd.models.transformer import LayerWeights, TransformerModel

pytestmark = pytest.mark.gpu
DEV, BF = torch.device("cuda"), torch.bfloat16


def _rnd(g, *shape, std=1.0, mean=0.0):
    return torch.empty(shape, dtype=BF, device=DEV).normal_(mean, std, generator=g)


# K: waves without a chunk, fewer chunks than the ring has stages, uneven shares; N: one tile, whole rounds, a second round of some tiles
@pytest.mark.parametrize("n,k", [(16, 64), (48, 448), (4096, 512), (4112, 576), (8192, 1088), (3072, 4096), (512, 14336)])
@pytest.mark.parametrize("m", [1, 7, 8, 9, 16])
def test_row_add(m, n, k):
    g = torch.Generator(device=DEV).manual_seed(n + k + m)
    x, w, res, norm = _rnd(g, m, k + 8)[:, :k], _rnd(g, n, k, std=k ** -0.5), _rnd(g, m, n), _rnd(g, n, std=0.2, mean=1)
    plain, new = res.clone(), res.clone()
    assert ops.row_add(x, w, plain, None) == (None, None)
    normed, squares = ops.row_add(x, w, new, norm)
    assert torch.equal(plain, new)
    want = x.double() @ w.double().t() + res.double()
    # the product and the sum are rounded to 8 bits each
    assert float((new.double() - want).abs().max() / want.abs().max()) < 2 ** -7
    assert float((new.double() - want).norm() / want.norm()) < 2 ** -8
    assert torch.equal(normed, (new.float() * norm.float()).to(BF))
    sums = new.double().square().view(m, n // 16, 16).sum(2)
    assert float((squares.double() - sums).abs().max() / sums.abs().max()) < 1e-6


@pytest.mark.parametrize("n_q,n_kv,k", [(32, 8, 4096), (28, 4, 3584), (52, 4, 512), (6, 1, 8192), (1, 1, 64)])
@pytest.mark.parametrize("m", [1, 8, 11])
@pytest.mark.parametrize("bias", [False, True])
def test_row_attention_projection(m, n_q, n_kv, k, bias):
    """Against the product in 64 bits, rounded, rotated and written by the passes that other batches take; decode attention over one page."""
    g = torch.Generator(device=DEV).manual_seed(n_q + k + m)
    n = (n_q + 2 * n_kv) * 128
    normed, w, b = _rnd(g, m, k), _rnd(g, n, k, std=k ** -0.5), _rnd(g, n) if bias else None
    squares = torch.rand(m, k // 16, device=DEV, generator=g) * 16
    cos_sin = ops.build_cos_sin(128, 256, 10000.0, device=DEV)
    meta = BatchMeta(positions=torch.arange(m, dtype=torch.int32, device=DEV) + 5,
                     slots=torch.arange(m, device=DEV) * 64 + torch.arange(m, device=DEV) + 5, num_decode=m)
    if m > 1:
        meta.slots[1] = -1
    meta.dec_block_tables, meta.dec_ctx_lens = torch.arange(m, dtype=torch.int32, device=DEV).view(m, 1), meta.positions + 1
    start = _rnd(g, m, 2, 2, n_kv, 64 * 128)
    got_pool, want_pool = start.clone(), start.clone()
    got = ops.row_attention_block((normed, squares), 1e-5, w, b, got_pool, 1, meta, n_q, n_kv, 128, 128 ** -0.5, cos_sin)
    factor = (squares.double().sum(1) / k + 1e-5).rsqrt()
    qkv = ((normed.double() @ w.double().t()) * factor[:, None] + (0 if b is None else b.double())).to(BF)
    want = ops.attention_block(qkv, want_pool, 1, meta, n_q, n_kv, 128, 128 ** -0.5, cos_sin)
    wrote = (want_pool != start).sum()
    assert wrote > 0 and abs(int((got_pool != start).sum()) - int(wrote)) <= 0.01 * int(wrote)
    # sums in 32 bits flip last places of 8 bits, before the rotation and behind it
    assert float((got_pool.float() - want_pool.float()).norm() / (want_pool.float() - start.float()).norm()) < 2 ** -8
    assert float((got.float() - want.float()).norm() / want.float().norm()) < 1e-2


@pytest.mark.parametrize("m,inter,k", [(1, 16384, 512), (14, 12288, 4096), (16, 16384, 8192)])
def test_row_gate_up(m, inter, k):
    g = torch.Generator(device=DEV).manual_seed(inter + m)
    normed, w = _rnd(g, m, k), _rnd(g, 2 * inter, k, std=k ** -0.5)
    squares = torch.rand(m, k // 16, device=DEV, generator=g) * 16
    h = (normed.double() @ w.double().t()) * (squares.double().sum(1) / k + 1e-5).rsqrt()[:, None]
    want = torch.nn.functional.silu(h[:, :inter]) * h[:, inter:]
    assert float((ops.row_gate_up((normed, squares), 1e-5, w).double() - want).norm() / want.norm()) < 2 ** -8


@pytest.mark.parametrize("grouped", [False, True])
@torch.inference_mode()
def test_decode_steps_with_and_without(monkeypatch, grouped):
    g = torch.Generator(device=DEV).manual_seed(3)
    h, inter, nq, nkv, layers = 3072, 12288, 24, 8, 4
    cfg = dataclasses.replace(PRESETS["llama-3-8b"], num_layers=layers, hidden_size=h, intermediate_size=inter, num_heads=nq, num_kv_heads=nkv, vocab_size=512)
    model = TransformerModel(cfg, BF, DEV, 1024)
    for _ in range(layers):
        lw = LayerWeights()
        lw.ln1, lw.ln2 = _rnd(g, h, std=0.2, mean=1), _rnd(g, h, std=0.2, mean=1)
        lw.wqkv, lw.wo = _rnd(g, (nq + 2 * nkv) * 128, h, std=0.02), _rnd(g, h, nq * 128, std=0.02)
        lw.w_gate_up, lw.w_down = _rnd(g, 2 * inter, h, std=0.02), _rnd(g, h, inter, std=0.02)
        model.layers.append(lw)
    model.embed, model.norm, model.lm_head = _rnd(g, 512, h), _rnd(g, h, std=0.2, mean=1), _rnd(g, 512, h, std=0.02)
    ctx = torch.tensor([1, 64, 65, 200, 1], dtype=torch.int32, device=DEV)
    table = torch.arange(20, dtype=torch.int32, device=DEV).view(5, 4)
    pos = ctx - 1
    slots = table.gather(1, (pos // 64).long()[:, None])[:, 0].long() * 64 + pos % 64
    slots[4] = -1
    meta = BatchMeta(positions=pos, slots=slots, num_decode=5, dec_block_tables=table, dec_ctx_lens=ctx)
    start = _rnd(g, 21, layers, 2, nkv, 64 * 128)
    ids = torch.arange(5, device=DEV) * 101
    taken = []
    real = ops.row_add
    monkeypatch.setattr(ops, "row_add", lambda *a: taken.append(a[3] is not None) or real(*a))

    def run():
        pool = ops.LayerGroupedPool([start[:, :2].clone(), start[:, 2:].clone()]) if grouped else start.clone()
        y = model.compute_logits(model.forward(ids, pool, meta))
        return y.double(), (torch.cat(pool.groups, 1) if grouped else pool).float()

    y, p = run()
    assert taken == [True, True] * (layers - 1) + [True, False]
    monkeypatch.setattr(ops, "ROW_ROWS", 4)  # (the batch has one row more)
    yw, pw = run()
    assert len(taken) == 2 * layers
    assert float((y - yw).norm() / yw.norm()) < 2e-2 and float((p - pw).norm() / (pw - start.float()).norm()) < 2e-2
    with torch.inference_mode(False), torch.enable_grad():
        model.layers[0].wo = model.layers[0].wo.clone().requires_grad_()
        assert not ops.row_layer_takes(_rnd(g, 3, h), model.layers[0], start, dataclasses.replace(meta, num_decode=3), nq, nkv, 128, model.cos_sin)
