"""Projections of up to a few hundred rows: row counts around tiles and row blocks, fewer chunks than stages, uneven splits, bias, the gated
unit, strided rows, and what the dispatch leaves to other kernels."""

import pytest
import torch

from vllm_production_stack_amd import ops

pytestmark = pytest.mark.gpu
DEV, BF = torch.device("cuda"), torch.bfloat16


@pytest.fixture
def any_shape(monkeypatch):
    monkeypatch.setattr(ops, "MID_MIN_FILL", 0.0)
    monkeypatch.setattr(ops, "MID_ROWS", ops.MID_ROWS_LONG)


@pytest.mark.parametrize("m", [1, 16, 17, 33, 48, 63, 80, 97, 112, 127, 128, 129, 200, 256])
@pytest.mark.parametrize("n,k,kind", [(128, 64, ""), (256, 192, "bias"), (128, 1088, ""), (256, 2624, "bias"), (384, 1088, "pair"), (256, 128, "pair"),
                                      # eight, nine and seventeen ranges of the reduction: its sums are read eight at a time
                                      (256, 4096, ""), (256, 4672, "bias"), (128, 8704, ""), (256, 4672, "pair"), (128, 8704, "pair")])
def test_matches_float64(any_shape, m, n, k, kind):
    g = torch.Generator(device=DEV).manual_seed(m + n + k)
    x = torch.randn(m, k + 8, generator=g, device=DEV).to(BF)[:, :k]   # rows of a wider tensor
    w = (torch.randn(n, k, generator=g, device=DEV) * k ** -0.5).to(BF)
    b = torch.randn(n, generator=g, device=DEV).to(BF) if kind == "bias" else None
    got = ops._mid_gemm(x, w, b, kind == "pair")
    assert got is not None
    if k >= 4096:
        assert ops._mid_splits(m, n, k, kind == "pair") == {4096: 8, 4672: 9, 8704: 17}[k]
    want = x.double() @ w.double().t()
    if kind == "pair":
        want = torch.nn.functional.silu(want[:, :n // 2]) * want[:, n // 2:]
    elif b is not None:
        want = want + b.double()
    # sums in 32 bits, one rounding to 16: half a unit in the last place, 2^-9, of every value
    assert float(((got.double() - want).abs() - want.abs() * 2 ** -8 - 1e-5).max()) < 0
    assert torch.equal(got, ops._mid_gemm(x, w, b, kind == "pair"))    # fixed order of the partial sums


def test_dispatch():
    w = torch.zeros(4096, 4096, device=DEV, dtype=BF)
    x = torch.zeros(300, 4096, device=DEV, dtype=BF)
    assert ops._mid_gemm(x[:40], w, None, False) is not None
    assert ops._mid_gemm(x[:120], w, None, False) is None              # partial sums of three quarters of the weights' bytes
    assert ops._mid_gemm(x, w, None, False) is None
    assert ops._mid_gemm(x[:40], w[:3584], None, False) is not None    # 224 workgroups
    assert ops._mid_gemm(x[:40], w[:2048], None, False) is None        # 128
    assert ops._mid_gemm(x[:40, 1:], w[:, 1:].contiguous(), None, False) is None   # a reduction that is no multiple of a chunk
    assert ops._mid_gemm(x[:40].float(), w, None, False) is None
    with torch.enable_grad():
        assert ops._mid_gemm(x[:40].clone().requires_grad_(), w, None, False) is None


@pytest.mark.parametrize("m", [96, 97, 112, 128])
def test_two_rounds_of_a_block_of_rows(m):
    """Two rounds of workgroups with 97 to 128 rows where the second is three quarters full (448 workgroups), not where it is half (400).
    Eight chunks: workgroups start at each of them."""
    g = torch.Generator(device=DEV).manual_seed(m)
    x = torch.randn(129, 512, generator=g, device=DEV).to(BF)
    w = (torch.randn(57344, 512, generator=g, device=DEV) * 512 ** -0.5).to(BF)
    got = ops._mid_gemm(x[:m], w, None, True)
    gu = x[:m].double() @ w.double().t()
    want = torch.nn.functional.silu(gu[:, :28672]) * gu[:, 28672:]
    assert float(((got.double() - want).abs() - want.abs() * 2 ** -8 - 1e-5).max()) < 0   # as above: one rounding to 16 bits
    assert (ops._mid_gemm(x[:m], w[:51200], None, True) is not None) == (m <= 96)
    assert ops._mid_gemm(x, w, None, True) is None


@pytest.mark.parametrize("m", [1, 24, 90])
def test_operands_on_another_device_are_refused(m):
    """A weight, bias or norm that still lies on the host raises, as in the library, and no kernel reads it."""
    x = torch.zeros(m, 4096, device=DEV, dtype=BF)
    w, b = torch.zeros(4096, 4096, device=DEV, dtype=BF), torch.zeros(4096, device=DEV, dtype=BF)
    for bad_w, bad_b in ((w.cpu(), None), (w.cpu(), b), (w, b.cpu())):
        with pytest.raises(RuntimeError):
            ops.linear(x, bad_w, bad_b)
    with pytest.raises(RuntimeError):
        ops.gate_up_silu(x, w.cpu())
    res = torch.zeros(m, 4096, device=DEV, dtype=BF)
    assert ops.linear_add_norm(x, w.cpu(), res, b, 1e-5) is None
    assert ops.linear_add_norm(x, w, res.cpu(), b, 1e-5) is None
    assert ops.linear_add_norm(x, w, res, b.cpu(), 1e-5) is None


@pytest.mark.filterwarnings("ignore::torch.jit.TracerWarning")
@pytest.mark.parametrize("m", [24, 90])
def test_calls_that_something_follows_stay_with_the_library(m):
    """Gradients of the bias alone, forward-mode tangents, vmap and traces, at rows where the kernel takes plain calls."""
    from torch.autograd import forward_ad

    g = torch.Generator(device=DEV).manual_seed(m)
    x, w = (torch.randn(n, 4096, generator=g, device=DEV).to(BF) for n in (m, 4096))
    b = torch.randn(4096, generator=g, device=DEV).to(BF)
    assert ops._mid_takes(x, w, b, False)
    lib = torch.nn.functional.linear
    with torch.enable_grad():
        leaf = b.clone().requires_grad_()
        ops.linear(x, w, leaf).sum().backward()
        assert torch.equal(leaf.grad, torch.full_like(b, m))
    with torch.no_grad(), forward_ad.dual_level():
        t = torch.randn(m, 4096, generator=g, device=DEV).to(BF)
        got = forward_ad.unpack_dual(ops.linear(forward_ad.make_dual(x, t), w, b)).tangent
        assert got is not None and torch.equal(got, lib(t, w))
    with torch.no_grad():
        xs = torch.stack([x, x.flip(0), -x])
        assert torch.func.vmap(lambda q: ops.linear(q, w))(xs).shape == (3, m, 4096)
        traced = torch.jit.trace(lambda q: ops.linear(q, w, b), (x,), check_trace=False)
        assert torch.equal(traced(xs[1]), lib(xs[1], w, b))
        ln = torch.func.vmap(lambda q: ops.layer_norm(q, b[:1024], b[1024:2048], 1e-5))(xs[..., :1024])
        assert torch.equal(ln, torch.nn.functional.layer_norm(xs[..., :1024], (1024,), b[:1024], b[1024:2048], 1e-5))


@pytest.mark.parametrize("tokens", [1, 2, 16, 17, 33, 49, 65, 130])
@pytest.mark.parametrize("routing", ["spread", "one expert"])
def test_experts(tokens, routing):
    """Expert row counts around the row tiles and the passes over an expert's weights, experts without rows."""
    g = torch.Generator(device=DEV).manual_seed(tokens)
    e, h, i, k = 4, 256, 512, 2
    x = torch.randn(tokens, h, generator=g, device=DEV).to(BF)
    w13 = (torch.randn(e, 2 * i, h, generator=g, device=DEV) * h ** -0.5).to(BF)
    w2 = (torch.randn(e, h, i, generator=g, device=DEV) * i ** -0.5).to(BF)
    first = torch.full((tokens,), 2, device=DEV) if routing == "one expert" else torch.randint(0, e, (tokens,), generator=g, device=DEV)
    ids = torch.stack([first, (first + 1) % e], 1).int()
    wt = torch.rand(tokens, k, generator=g, device=DEV)
    got = ops.moe_experts_grouped(x, w13, w2, ids, wt)
    want = torch.zeros(tokens, h, dtype=torch.float64, device=DEV)
    for j in range(k):
        gu = torch.stack([w13[c].double() @ x[t].double() for t, c in enumerate(ids[:, j].tolist())])
        act = torch.nn.functional.silu(gu[:, :i]) * gu[:, i:]
        want += wt[:, j:j + 1].double() * torch.stack([w2[c].double() @ act[t] for t, c in enumerate(ids[:, j].tolist())])
    # activations, unit outputs and result rounded to 16 bits: 2^-9 of the norm each
    assert float((got.double() - want).norm() / want.norm()) < 6e-3


def test_experts_of_a_large_batch():
    """Rows of the activations beyond the first 4 GiB: an early and a late expert's tokens against float64."""
    g = torch.Generator(device=DEV).manual_seed(3)
    e, h, i, t = 4, 128, 16384, 65600
    x = torch.randn(t, h, generator=g, device=DEV).to(BF)
    w13 = (torch.randn(e, 2 * i, h, generator=g, device=DEV) * h ** -0.5).to(BF)
    w2 = (torch.randn(e, h, i, generator=g, device=DEV) * i ** -0.5).to(BF)
    ids = torch.stack([torch.arange(t, device=DEV) % e, (torch.arange(t, device=DEV) + 1) % e], 1).int()
    wt = torch.rand(t, 2, generator=g, device=DEV)
    got = ops.moe_experts_grouped(x, w13, w2, ids, wt)
    for row in (0, 1, 2, 3, 30000, t - 4, t - 3, t - 2, t - 1):
        want = torch.zeros(h, dtype=torch.float64, device=DEV)
        for c, p in zip(ids[row].tolist(), wt[row].double()):
            gu = w13[c].double() @ x[row].double()
            want += p * (w2[c].double() @ (torch.nn.functional.silu(gu[:i]) * gu[i:]))
        assert float((got[row].double() - want).norm() / want.norm()) < 6e-3   # as above


def test_an_expert_beyond_four_gigabytes():
    g = torch.Generator(device=DEV).manual_seed(5)
    h, i = 16384, 65536 + 512
    x = torch.randn(3, h, generator=g, device=DEV).to(BF)
    w13 = torch.empty(1, 2 * i, h, device=DEV, dtype=BF).normal_(0, h ** -0.5, generator=g)
    w2 = torch.empty(1, h, i, device=DEV, dtype=BF).normal_(0, i ** -0.5, generator=g)
    got = ops.moe_experts_grouped(x, w13, w2, torch.zeros(3, 1, dtype=torch.int32, device=DEV), torch.ones(3, 1, device=DEV))
    gu = torch.cat([x.float() @ c.float().t() for c in w13[0].split(16384)], 1)
    act = torch.nn.functional.silu(gu[:, :i]) * gu[:, i:]
    want = torch.cat([act @ c.float().t() for c in w2[0].split(4096)], 1)
    assert float((got.float() - want).norm() / want.norm()) < 6e-3   # as above


def test_experts_off_the_16_byte_boundary():
    """Weights and rows that start two bytes into a buffer give what aligned copies give."""
    g = torch.Generator(device=DEV).manual_seed(4)

    def odd(*shape):
        n = torch.Size(shape).numel()
        return (torch.randn(n + 1, generator=g, device=DEV) * 0.1).to(BF)[1:].view(shape)

    x, w13, w2 = odd(20, 256), odd(4, 1024, 256), odd(4, 256, 512)
    ids = torch.randint(0, 4, (20, 1), generator=g, device=DEV, dtype=torch.int32)
    wt = torch.ones(20, 1, device=DEV)
    assert torch.equal(ops.moe_experts_grouped(x, w13, w2, ids, wt), ops.moe_experts_grouped(x.clone(), w13.clone(), w2.clone(), ids, wt))


@pytest.mark.parametrize("m,n,k", [(1, 256, 1024), (3, 1280, 1088), (16, 4096, 1024), (17, 5120, 1088), (40, 8192, 2624), (130, 128, 1088),
                                   (5, 256, 4096), (3, 256, 4672), (17, 384, 8704)])
def test_sum_with_residual_and_norm(any_shape, m, n, k):
    """One reduction against the separate passes: the same roundings, so the residual stream is equal and the norm differs by its
    sum of squares' order (one unit in the last place of 16 bits)."""
    g = torch.Generator(device=DEV).manual_seed(m + n + k)
    x = torch.randn(m, k, generator=g, device=DEV).to(BF)
    w = (torch.randn(n, k, generator=g, device=DEV) * k ** -0.5).to(BF)
    res, ln = torch.randn(m, n, generator=g, device=DEV).to(BF), torch.randn(n, generator=g, device=DEV).to(BF)
    want_res = res.clone()
    want = ops.rms_norm(ops._mid_gemm(x, w, None, False), ln, 1e-5, want_res)
    got = ops.linear_add_norm(x, w, res, ln, 1e-5)
    assert got is not None and torch.equal(res, want_res)
    assert float(((got.float() - want.float()).abs() - want.float().abs() * 2 ** -7).max()) <= 0
    kept = res.clone()
    assert ops.linear_add_norm(x[:, 1:], w[:, 1:].contiguous(), res, ln, 1e-5) is None and torch.equal(res, kept)


@pytest.mark.parametrize("m", [96, 97, 112, 128])
def test_sum_with_norm_of_a_block_of_rows(m):
    """Partial sums of up to the weights' bytes (128 rows in eight ranges) where the reduction makes the norm, three quarters elsewhere."""
    g = torch.Generator(device=DEV).manual_seed(m)
    x = torch.randn(129, 4096, generator=g, device=DEV).to(BF)
    w = (torch.randn(4096, 4096, generator=g, device=DEV) / 64).to(BF)
    res, ln = torch.randn(129, 4096, generator=g, device=DEV).to(BF), torch.randn(4096, generator=g, device=DEV).to(BF)
    got_res, kept = res[:m].clone(), res.clone()
    got = ops.linear_add_norm(x[:m], w, got_res, ln, 1e-5)
    assert got is not None and (ops._mid_gemm(x[:m], w, None, False) is not None) == (m <= 96)
    assert ops.linear_add_norm(x, w, res, ln, 1e-5) is None and torch.equal(res, kept)
    add = x[:m].double() @ w.double().t()
    want = add + res[:m].double()
    # two roundings to 16 bits, of the sum and of the new row: half a unit in the last place, 2^-9, of each and the first's share again
    assert float(((got_res.double() - want).abs() - 2 ** -8 * (add.abs() + want.abs()) - 1e-5).max()) < 0
    norm = got_res.double() * (got_res.double().square().mean(1, keepdim=True) + 1e-5).rsqrt() * ln.double()
    assert float(((got.double() - norm).abs() - 2 ** -8 * norm.abs() - 1e-5).max()) < 0


@pytest.mark.parametrize("m,n_q,n_kv,bias,k", [(1, 32, 8, False, 1088), (3, 5, 1, True, 1088), (17, 8, 8, True, 1088), (40, 32, 8, False, 1088),
                                               (5, 2, 1, False, 4096), (3, 2, 1, True, 4672), (17, 4, 1, False, 8704)])
def test_sum_with_rotation_and_cache_write(any_shape, m, n_q, n_kv, bias, k):
    """Query rows and the pages that a decode step's projection leaves against the separate passes, one row without a slot."""
    g = torch.Generator(device=DEV).manual_seed(m)
    n = (n_q + 2 * n_kv) * 128
    x = torch.randn(m, k, generator=g, device=DEV).to(BF)
    w = (torch.randn(n, k, generator=g, device=DEV) * k ** -0.5).to(BF)
    b = torch.randn(n, generator=g, device=DEV).to(BF) if bias else None
    pages = m + 2
    pool = torch.randn(pages, 2, 2, n_kv * 64 * 128, generator=g, device=DEV).to(BF)
    positions = torch.randint(0, 500, (m,), generator=g, device=DEV, dtype=torch.int32)
    slots = torch.randperm(pages * 64, generator=g, device=DEV)[:m]
    slots[m // 2] = slots[m // 2] if m == 1 else -1
    ang = torch.rand(500, 64, generator=g, device=DEV) * 6.28
    cos_sin = torch.cat([ang.cos(), ang.sin()], dim=1).contiguous()
    want_pool, qkv = pool.clone(), ops._mid_gemm(x, w, b, False)
    ops.rope_and_cache(qkv, positions, slots, cos_sin, want_pool, 1, n_q, n_kv, 128)
    q = ops.decode_qkv(x, w, b, pool, 1, positions, slots, cos_sin, n_q, n_kv)
    assert torch.equal(q, qkv[:, :n_q * 128]) and torch.equal(pool, want_pool)


def _decoder(layers, g):
    import dataclasses

    from vllm_production_stack_amd.engine.config import PRESETS
    from vllm_production_stack_amd.models.transformer import LayerWeights, TransformerModel

    cfg = dataclasses.replace(PRESETS["llama-3-8b"], num_layers=layers, hidden_size=1024, intermediate_size=2048, num_heads=8,
                              num_kv_heads=2, vocab_size=1024)
    h, i, d = cfg.hidden_size, cfg.intermediate_size, cfg.head_dim
    model = TransformerModel(cfg, BF, DEV, 1024)

    def rnd(*shape, std=None):
        return torch.empty(shape, device=DEV, dtype=BF).normal_(0, std or shape[-1] ** -0.5, generator=g)

    for _ in range(layers):
        lw = LayerWeights()
        lw.ln1, lw.ln2 = rnd(h, std=0.3) + 1, rnd(h, std=0.3) + 1
        lw.wqkv, lw.wo = rnd((cfg.num_heads + 2 * cfg.num_kv_heads) * d, h), rnd(h, cfg.num_heads * d)
        lw.w_gate_up, lw.w_down = rnd(2 * i, h), rnd(h, i)
        model.layers.append(lw)
    model.embed, model.norm, model.lm_head = rnd(cfg.vocab_size, h, std=1), rnd(h, std=0.3) + 1, rnd(cfg.vocab_size, h)
    return cfg, model


@pytest.mark.parametrize("grouped", [False, True])
@torch.inference_mode()
def test_decoder_steps_with_the_fused_reductions(monkeypatch, grouped):
    """A decode step (one row without a slot, as in a padded graph) and a short prefill of three layers, with the reductions that also
    update the residual stream, make the norm, rotate and write the cache, against the separate passes."""
    from vllm_production_stack_amd.models.batch import BatchMeta

    g = torch.Generator(device=DEV).manual_seed(11)
    layers = 4 if grouped else 3
    cfg, model = _decoder(layers, g)
    nq, nkv, d = cfg.num_heads, cfg.num_kv_heads, cfg.head_dim
    ctx = [1, 64, 65, 200, 300, 1]
    table = torch.arange(6 * 5, dtype=torch.int32, device=DEV).view(6, 5)
    start = torch.randn(31, layers, 2, nkv, 64 * d, generator=g, device=DEV).to(BF)

    def pool():
        return ops.LayerGroupedPool([start[:, :2].clone(), start[:, 2:].clone()]) if grouped else start.clone()

    pos = torch.tensor([c - 1 for c in ctx], dtype=torch.int32, device=DEV)
    slots = table.gather(1, (pos // 64).long()[:, None])[:, 0].long() * 64 + pos % 64
    slots[5] = -1
    decode = BatchMeta(positions=pos, slots=slots, num_decode=6)
    decode.dec_block_tables, decode.dec_ctx_lens = table, pos + 1
    decode.dec_num_splits = 3
    lens, total = [13, 40], 53
    pre = BatchMeta(positions=torch.cat([torch.arange(n, dtype=torch.int32) for n in lens]).to(DEV),
                    slots=torch.cat([torch.arange(s * 320, s * 320 + n) for s, n in enumerate(lens)]).to(DEV))
    pre.num_prefill_seqs, pre.pre_block_tables = 2, table[:2].contiguous()
    pre.pre_ctx_lens = torch.tensor(lens, dtype=torch.int32, device=DEV)
    pre.pre_cu_q = torch.tensor([0, 13, 53], dtype=torch.int32, device=DEV)
    pre.pre_tile_rows = ops.prefill_tile_rows(lens, nq, nkv)
    ts, tq = ops.build_prefill_tiles(lens, nq, nkv, pre.pre_tile_rows, lens)
    pre.pre_tile_seq, pre.pre_tile_q0 = (torch.tensor(v, dtype=torch.int32, device=DEV) for v in (ts, tq))

    def run(meta, rows):
        p = pool()
        ids = torch.arange(rows, device=DEV) * 17 % cfg.vocab_size
        y = model.compute_logits(model.forward(ids, p, meta))
        return y.float(), (torch.cat(p.groups, 1) if grouped else p).float()

    was = ops.set_skinny_gemm(False)
    want = [run(decode, 6), run(pre, total)]
    ops.set_skinny_gemm(was)
    monkeypatch.setattr(ops, "MID_MIN_FILL", 0.0)
    taken = {"linear_add_norm": 0, "decode_attention_block": 0}
    for name in taken:
        def spy(*args, _name=name, _real=getattr(ops, name), **kw):
            r = _real(*args, **kw)
            taken[_name] += r is not None
            return r
        monkeypatch.setattr(ops, name, spy)
    got = [run(decode, 6)]
    assert taken == {"linear_add_norm": 2 * layers - 1, "decode_attention_block": layers}   # (the last down projection has no norm behind it)
    got.append(run(pre, total))
    assert taken == {"linear_add_norm": 2 * (2 * layers - 1), "decode_attention_block": layers}
    for (y, p), (yw, pw) in zip(got, want):
        # sums in another order flip last places of 16 bits, 2^-8 of a value at most (a cached entry), and three or four layers
        # pass them on: 0.7 to 0.9 % of the logits' norm
        assert float((y - yw).norm() / yw.norm()) < 2e-2
        assert float((p - pw).norm() / pw.norm()) < 2 ** -8
    untouched = torch.ones(31, dtype=torch.bool, device=DEV)
    untouched[(slots[:5] // 64)] = False
    assert torch.equal(got[0][1][untouched], start.float()[untouched])                      # nothing went to the row without a slot


@pytest.mark.filterwarnings("ignore::torch.jit.TracerWarning")
@pytest.mark.parametrize("m,n,k", [(1, 520, 512), (8, 2048, 2048), (16, 256, 4096), (40, 1024, 8192)])
def test_followed_calls_of_few_rows(m, n, k):
    """Gradients, tangents, vmap and traces where the streaming kernels are the ones that take the size, plain, gated and of a packed copy."""
    from torch.autograd import forward_ad

    g = torch.Generator(device="cuda").manual_seed(m)
    x, t = (torch.randn(m, k, generator=g, device="cuda").to(torch.bfloat16) for _ in range(2))
    w = (torch.randn(n, k, generator=g, device="cuda") * k ** -0.5).to(torch.bfloat16)
    lib = torch.nn.functional.linear
    packed = ops.pack_weight(w) if ops.packed_supported(n, k) else None
    with torch.enable_grad():
        for call in (lambda a: ops.linear(a, w), lambda a: ops.gate_up_silu(a, w), lambda a: ops.linear(a, w, None, packed)):
            leaf = x.clone().requires_grad_()
            call(leaf).sum().backward()
            assert leaf.grad is not None and float(leaf.grad.float().norm()) > 0
    with torch.no_grad(), forward_ad.dual_level():
        assert torch.equal(forward_ad.unpack_dual(ops.linear(forward_ad.make_dual(x, t), w)).tangent, lib(t, w))
    with torch.no_grad():
        xs = torch.stack([x, t])
        assert torch.func.vmap(lambda q: ops.linear(q, w))(xs).shape == (2, m, n)
        assert torch.func.vmap(lambda q: ops.gate_up_silu(q, w))(xs).shape == (2, m, n // 2)
        traced = torch.jit.trace(lambda q: ops.linear(q, w), (x,), check_trace=False)
        assert torch.equal(traced(t), lib(t, w))
