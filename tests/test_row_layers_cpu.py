"""Which layers of a decode step take the products of a few rows: each that fits, whatever stands before it."""

import dataclasses

import pytest
import torch

from vllm_production_stack_amd import ops
from vllm_production_stack_amd.engine.config import PRESETS
from vllm_production_stack_amd.models.batch import BatchMeta
from vllm_production_stack_amd.models.transformer import LayerWeights, TransformerModel


@pytest.mark.parametrize("fits", ["1111", "0000", "1011", "0110", "1001", "0101"])
@torch.inference_mode()
def test_every_layer_that_fits(monkeypatch, fits):
    g = torch.Generator().manual_seed(3)
    h, inter, nq, nkv, d, layers, rows = 64, 96, 4, 2, 16, 4, 3
    rnd = lambda *shape, std=1.0, mean=0.0: torch.empty(shape).normal_(mean, std, generator=g)  # noqa: E731
    cfg = dataclasses.replace(PRESETS["llama-3-8b"], num_layers=layers, hidden_size=h, intermediate_size=inter, num_heads=nq, num_kv_heads=nkv, head_dim=d,
                              vocab_size=50)
    model = TransformerModel(cfg, torch.float32, torch.device("cpu"), 256)
    for _ in range(layers):
        lw = LayerWeights()
        lw.ln1, lw.ln2 = rnd(h, std=0.2, mean=1), rnd(h, std=0.2, mean=1)
        lw.wqkv, lw.wo = rnd((nq + 2 * nkv) * d, h, std=0.1), rnd(h, nq * d, std=0.1)
        lw.w_gate_up, lw.w_down = rnd(2 * inter, h, std=0.1), rnd(h, inter, std=0.1)
        model.layers.append(lw)
    model.embed, model.norm, model.lm_head = rnd(50, h), rnd(h, std=0.2, mean=1), rnd(50, h, std=0.1)
    pos = torch.tensor([5, 63, 70], dtype=torch.int32)
    table = torch.arange(6, dtype=torch.int32).view(3, 2)
    slots = table.gather(1, (pos // 64).long()[:, None])[:, 0].long() * 64 + pos % 64
    meta = BatchMeta(positions=pos, slots=slots, num_decode=rows, dec_block_tables=table, dec_ctx_lens=pos + 1)
    start, ids = rnd(6, layers, 2, nkv, 64 * d), torch.arange(rows) * 7
    added, attended = [], []

    def takes(residual, lw, *_):
        return fits[model.layers.index(lw)] == "1"

    def normed(rows, eps):
        return rows[0] * (rows[1].sum(1, keepdim=True) / h + eps).rsqrt()

    def row_add(x, w, residual, norm):
        added.append([next(i for i, lw in enumerate(model.layers) if w is lw.wo or w is lw.w_down), norm is not None])
        residual += x @ w.t()
        return (None, None) if norm is None else (residual * norm, residual.square().view(rows, -1, 16).sum(2))

    def row_attention_block(rows, eps, w, bias, pool, layer, *args):
        attended.append(layer)
        return ops.attention_block(torch.nn.functional.linear(normed(rows, eps), w, bias), pool, layer, *args)

    run = lambda pool: model.compute_logits(model.forward(ids, pool, meta))  # noqa: E731
    want_pool, got_pool = start.clone(), start.clone()
    want = run(want_pool)
    monkeypatch.setattr(ops, "row_layer_takes", takes)
    monkeypatch.setattr(ops, "row_add", row_add)
    monkeypatch.setattr(ops, "row_gate_up", lambda rows, eps, w: ops.silu_and_mul(torch.nn.functional.linear(normed(rows, eps), w)))
    monkeypatch.setattr(ops, "row_attention_block", row_attention_block)
    torch.testing.assert_close(run(got_pool), want, rtol=1e-4, atol=1e-4)
    torch.testing.assert_close(got_pool, want_pool, rtol=1e-4, atol=1e-4)
    behind = [fits[i + 1:i + 2] == "1" for i in range(layers)]  # a layer that fits makes the next one's norm only where that fits as well
    assert added == [v for i in range(layers) if fits[i] == "1" for v in ([i, True], [i, behind[i]])]
    assert attended == [i for i in range(1, layers) if fits[i - 1:i + 1] == "11"]
    monkeypatch.setattr(ops, "ROW_ROWS", rows - 1)
    added.clear()
    torch.testing.assert_close(run(start.clone()), want, rtol=0, atol=0)
    assert not added
