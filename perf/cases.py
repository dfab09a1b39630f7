"""What a replica of this stack spends its GPU time on, as cases that can be timed and checked.

A case is a dict of plain values.  ``listed()`` gives the fixed ones, ``draw(rng)`` more of the same ranges,
``prepare(case, seed)`` what a program holds before the call (weights, cache, work lists, captured graphs), ``run(state)``
one pass, ``work(case)`` the bytes and operations it cannot do without, ``exact(case, seed)`` the same outputs in 64 bits
from plain torch.  Kinds:

decode      one token for every running sequence of a decoder over its paged cache, as a captured graph (the way the
            engine runs decode steps): one user's stream, a few users, the 40 users with 21.5k-token histories of the
            multi-round question answering benchmark; routed mixtures too.
turn        the prompt of a new turn behind a cached history (up to 512 rows, a captured graph): time to first token of a
            conversation's next question.
prefill     a chunk of a prompt without a graph, up to the engine's 8192 rows a step, with or without cached tokens before
            it; routed mixtures too.
latent      attention of the latent-cache decoders (32 or 16 heads, entries of 512 + 64 channels): a decode batch, or a
            chunk of query rows.
scan        the recurrences with per-sequence state over prompt chunks: retention (fixed decays, rotated keys) and gated
            linear attention, state carried out in the sequences' slots.
speech      the Whisper encoder over 30 s windows, one request or a batch of them.
kv_encode   KV pages to the compressed form that the disk and remote tiers store (quantiser, entropy coder, to the host).
kv_decode   the way back, from stored bytes to pages on the GPU.

Decoders have the widths of the named presets and random weights; a few of their equal layers are kept (a step of all of
them is the same launches more often) so that three states fit the card.
"""

from __future__ import annotations

import dataclasses
import math

import numpy as np
import torch

from vllm_production_stack_amd import ops
from vllm_production_stack_amd.engine.config import PRESETS
from vllm_production_stack_amd.kv.serde import PageSerde, default_levels
from vllm_production_stack_amd.models.batch import BatchMeta
from vllm_production_stack_amd.models.transformer import LayerWeights, TransformerModel
from vllm_production_stack_amd.models.whisper import WHISPER_PRESETS, WhisperModel

PAGE = 64
MAX_LEN = 32768          # the engine's max_model_len for these presets
BF16 = torch.bfloat16
DEV = torch.device("cuda")


# ------------------------------------------------------------------------------------------------ the cases
def listed():
    return [
        # one user's stream: launches and the rate at which weights arrive
        {"name": "decode_1", "kind": "decode", "model": "llama-3-8b", "layers": 16, "batch": 1, "context": 2048},
        # a few users, contexts of different lengths, a batch that is no power of two
        {"name": "decode_12", "kind": "decode", "model": "llama-3-8b", "layers": 16, "batch": 12, "context": 2900},
        # the multi-round benchmark's decode steps: 40 users, 21.5k-token histories
        {"name": "decode_40_long", "kind": "decode", "model": "llama-3-8b", "layers": 8, "batch": 40, "context": 21500},
        # the benchmark's next question behind a history that is still cached
        {"name": "turn_97", "kind": "turn", "model": "llama-3-8b", "layers": 16, "rows": 97, "seqs": 1, "cached": 20900},
        # a cold history, one full engine chunk
        {"name": "prefill_8192", "kind": "prefill", "model": "llama-3-8b", "layers": 4, "rows": 8192, "seqs": 1, "cached": 0},
        # routed mixture: decode batch, and a chunk of an odd size from two prompts
        {"name": "moe_decode_8", "kind": "decode", "model": "mixtral-8x7b", "layers": 2, "batch": 8, "context": 2048},
        {"name": "moe_prefill_1531", "kind": "prefill", "model": "mixtral-8x7b", "layers": 2, "rows": 1531, "seqs": 2, "cached": 0},
        # latent-cache decoder: a decode batch at the architecture comparison's larger size
        {"name": "latent_32", "kind": "latent", "mode": "decode", "heads": 32, "batch": 32, "context": 4096},
        # retention layer over two prompts of the architecture comparison
        {"name": "retention_8192", "kind": "scan", "mode": "retention", "heads": 32, "rows": 8192, "seqs": 2},
        # a batch of speech requests
        {"name": "speech_8", "kind": "speech", "model": "whisper-small", "windows": 8},
        # pages of a finished prompt chunk going to the remote tier, and pages of a history coming back
        {"name": "kv_encode_4", "kind": "kv_encode", "model": "llama-3-8b", "pages": 4},
        {"name": "kv_decode_12", "kind": "kv_decode", "model": "llama-3-8b", "pages": 12},
    ]


def _log(rng, lo, hi):
    return int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))


def draw(rng):
    kind = rng.choice(["decode", "decode", "turn", "prefill", "moe_decode", "moe_prefill", "latent", "latent", "scan", "scan",
                       "speech", "kv_encode", "kv_decode"])
    if kind == "decode":  # up to the engine's 256 sequences, together at most the listed long batch's cache
        batch = _log(rng, 1, 256)
        return {"kind": "decode", "model": "llama-3-8b", "layers": 8, "batch": batch,
                "context": _log(rng, 64, min(24000, 860000 // batch))}
    if kind == "turn":
        seqs = rng.choice([1, 1, 1, 2, 3])
        return {"kind": "turn", "model": "llama-3-8b", "layers": 8, "rows": _log(rng, 16, 512), "seqs": seqs,
                "cached": _log(rng, 512, 30000 // seqs)}
    if kind == "prefill":
        cached = rng.choice([0, 0, _log(rng, 500, 12000)])
        return {"kind": "prefill", "model": "llama-3-8b", "layers": 4, "rows": _log(rng, 513, 3000 if cached else 8000),
                "seqs": rng.choice([1, 1, 2, 4]), "cached": cached}
    if kind == "moe_decode":
        return {"kind": "decode", "model": "mixtral-8x7b", "layers": 2, "batch": _log(rng, 1, 64), "context": _log(rng, 64, 6000)}
    if kind == "moe_prefill":
        return {"kind": "prefill", "model": "mixtral-8x7b", "layers": 2, "rows": _log(rng, 65, 6000),
                "seqs": rng.choice([1, 2, 3]), "cached": 0}
    if kind == "latent":
        heads = rng.choice([16, 32])
        if rng.random() < 0.6:
            batch = _log(rng, 1, 128)
            return {"kind": "latent", "mode": "decode", "heads": heads, "batch": batch, "context": _log(rng, 100, min(30000, 400000 // batch))}
        return {"kind": "latent", "mode": "prefill", "heads": heads, "batch": _log(rng, 20, 2000), "context": _log(rng, 2000, 8000)}
    if kind == "scan":
        seqs = rng.choice([1, 2, 3, 5, 8])
        return {"kind": "scan", "mode": rng.choice(["retention", "gated"]), "heads": rng.choice([16, 32]),
                "rows": _log(rng, 64 * seqs, 8192), "seqs": seqs}
    if kind == "speech":
        return {"kind": "speech", "model": rng.choice(["whisper-base", "whisper-small"]), "windows": _log(rng, 1, 32)}
    return {"kind": kind, "model": rng.choice(["llama-3-8b", "llama-3-70b", "qwen2.5-7b"]), "pages": rng.randint(1, 8)}


# ------------------------------------------------------------------------------------------------ inputs from the seed
def _gen(seed, *tags):
    x = (seed * 0x9E3779B1 + 0x1234567) & 0x7FFFFFFF
    for t in tags:
        x = ((x ^ (t + 0x51ED27)) * 0x85EBCA77 + 0x165667B1) & 0x7FFFFFFF
    return torch.Generator(device=DEV).manual_seed(x)


def _normal(g, *shape, std=1.0, mean=0.0, dtype=BF16):
    return torch.empty(shape, dtype=dtype, device=DEV).normal_(mean, std, generator=g)


def _config(case):
    return dataclasses.replace(PRESETS[case["model"]], num_layers=case["layers"])


# projections into the residual stream start smaller, by the root of the sublayers of a 32-layer decoder
INTO_STREAM = 0.02 / 64 ** 0.5


def _layer(cfg, seed, li):
    g = _gen(seed, 11, li)
    h, i, d = cfg.hidden_size, cfg.intermediate_size, cfg.head_dim
    w = {"ln1": _normal(g, h, std=0.1, mean=1.0), "ln2": _normal(g, h, std=0.1, mean=1.0),
         "wqkv": _normal(g, (cfg.num_heads + 2 * cfg.num_kv_heads) * d, h, std=0.02),
         "wo": _normal(g, h, cfg.num_heads * d, std=INTO_STREAM)}
    if cfg.num_experts:
        w["router"] = _normal(g, cfg.num_experts, h, std=0.02)
        w["w13"] = _normal(g, cfg.num_experts, 2 * i, h, std=0.02)
        w["w2"] = _normal(g, cfg.num_experts, h, i, std=INTO_STREAM)
    else:
        w["w_gate_up"] = _normal(g, 2 * i, h, std=0.02)
        w["w_down"] = _normal(g, h, i, std=INTO_STREAM)
    return w


def _ends(cfg, seed):
    g = _gen(seed, 12)
    h = cfg.hidden_size
    return {"embed": _normal(g, cfg.vocab_size, h), "norm": _normal(g, h, std=0.1, mean=1.0),
            "lm_head": _normal(g, cfg.vocab_size, h, std=0.02)}


def _history(cfg, seed, layer, seq, n):
    """Cached keys | values of a sequence's first n tokens, [n, 2 * kv heads * channels]."""
    return _normal(_gen(seed, 13, layer, seq), n, 2 * cfg.num_kv_heads * cfg.head_dim)


def _sequences(case):
    """(cached tokens, new tokens) of every sequence of the step."""
    if case["kind"] == "decode":  # contexts between three quarters and all of the stated one
        c = case["context"]
        return [(c - 1 - (i * 37) % (c // 4 + 1), 1) for i in range(case["batch"])]
    n, s = case["rows"], case["seqs"]
    cuts = [n * (3 * k + k * k) // (3 * s + s * s) for k in range(s + 1)]  # later prompts are longer
    return [(case["cached"] - 17 * k if case["cached"] else 0, cuts[k + 1] - cuts[k]) for k in range(s)]


def _tokens(cfg, seed, n):
    return torch.randint(0, cfg.vocab_size, (n,), device=DEV, generator=_gen(seed, 14))


def _levels(case):
    return default_levels(PRESETS[case["model"]].num_layers)


def _page(case, seed, i):
    """One KV page, [layer][K | V][kv head][64 x channels]: keys whose channels have a level of their own over the page's
    tokens (what the codec's anchors are for), values without."""
    cfg = PRESETS[case["model"]]
    g = _gen(seed, 15, i)
    rows = cfg.num_kv_heads * PAGE * cfg.head_dim // (32 * 64)
    k = _normal(g, cfg.num_layers, rows, 1, 64, std=1.5, dtype=torch.float32) + _normal(
        g, cfg.num_layers, rows, 32, 64, std=0.6, dtype=torch.float32)
    v = _normal(g, cfg.num_layers, rows, 32, 64, std=0.8, dtype=torch.float32)
    return torch.stack([k, v], dim=1).to(BF16).view(-1)


def _latent_inputs(case, seed):
    g = _gen(seed, 16)
    h = case["heads"]
    if case["mode"] == "decode":
        ctx = [c + n for c, n in _sequences({"kind": "decode", "batch": case["batch"], "context": case["context"]})]
        rows, seq, pos = len(ctx), list(range(len(ctx))), [c - 1 for c in ctx]
    else:  # a chunk at the end of one context
        rows, ctx = case["batch"], [case["context"]]
        seq, pos = [0] * rows, list(range(case["context"] - rows, case["context"]))
    pages = [-(-c // PAGE) for c in ctx]
    pool = _normal(g, sum(pages), PAGE * 576, std=0.5)
    order = torch.randperm(sum(pages), device=DEV, generator=g).int().tolist()
    table, at = [], 0
    for p in pages:
        table.append(order[at:at + p] + [0] * (max(pages) - p))
        at += p
    return {"q_lat": _normal(g, rows, h, 512, std=0.7), "q_rot": _normal(g, rows, h, 64, std=0.7), "pool": pool,
            "sink": _normal(g, h, dtype=torch.float32), "ctx": ctx, "seq": seq, "pos": pos, "table": table}


LATENT_SCALE = 192 ** -0.5


def _scan_lens(case):
    return [n for _, n in _sequences({"kind": "prefill", "rows": case["rows"], "seqs": case["seqs"], "cached": 0})]


def _scan_inputs(case, seed):
    g = _gen(seed, 17)
    h, retention = case["heads"], case["mode"] == "retention"
    vdim = 256 if retention else 128
    x = {"dim": 128, "vdim": vdim, "proj": _normal(g, case["rows"], h * (256 + vdim))}
    if retention:
        x["decay"] = [1 - 2.0 ** (-5 - 3 * i / h) for i in range(h)]
    else:
        x["bias"] = _normal(g, h * 128, std=0.5, mean=2.0, dtype=torch.float32)
        x["lower"] = torch.empty(h * 128, device=DEV).uniform_(0.2, 0.9, generator=g)
    return x


def _speech_weights(case, seed):
    c = WHISPER_PRESETS[case["model"]]
    g = _gen(seed, 18)
    d, f = c.d_model, c.encoder_ffn_dim
    w = {"encoder.conv1.weight": _normal(g, d, c.num_mel_bins, 3, std=0.08), "encoder.conv1.bias": _normal(g, d, std=0.05),
         "encoder.conv2.weight": _normal(g, d, d, 3, std=0.02), "encoder.conv2.bias": _normal(g, d, std=0.05),
         "encoder.embed_positions.weight": _normal(g, c.max_source_positions, d, std=0.5)}

    def norm(name):
        w[name + ".weight"], w[name + ".bias"] = _normal(g, d, std=0.1, mean=1.0), _normal(g, d, std=0.05)

    def linear(name, n, k, bias=True):
        w[name + ".weight"] = _normal(g, n, k, std=k ** -0.5)
        if bias:
            w[name + ".bias"] = _normal(g, n, std=0.05)

    for i in range(c.encoder_layers):
        p = f"encoder.layers.{i}."
        norm(p + "self_attn_layer_norm")
        for proj in ("q_proj", "k_proj", "v_proj", "out_proj"):
            linear(p + "self_attn." + proj, d, d, proj != "k_proj")
        norm(p + "final_layer_norm")
        linear(p + "fc1", f, d)
        linear(p + "fc2", d, f)
    norm("encoder.layer_norm")
    return w


def _mel(case, seed):  # log-mel values lie between about -1 and 1
    c = WHISPER_PRESETS[case["model"]]
    return _normal(_gen(seed, 19), case["windows"], c.num_mel_bins, 2 * c.max_source_positions, dtype=torch.float32).tanh()


# ------------------------------------------------------------------------------------------------ what a program holds
def _dev(values, dtype):
    return torch.tensor(values, dtype=dtype, device=DEV)


def _captured(step):
    """A graph of ``step`` and its output, the way the engine captures its steps."""
    side = torch.cuda.Stream()
    side.wait_stream(torch.cuda.current_stream())
    with torch.cuda.stream(side):
        step()
    torch.cuda.current_stream().wait_stream(side)
    torch.cuda.synchronize()
    graph = torch.cuda.CUDAGraph()
    with torch.cuda.graph(graph):
        out = step()
    return graph, out


def _prepare_decoder(case, seed):
    cfg = _config(case)
    model = TransformerModel(cfg, BF16, DEV, MAX_LEN)
    ends = _ends(cfg, seed)
    model.embed, model.norm, model.lm_head = ends["embed"], ends["norm"], ends["lm_head"]
    for li in range(cfg.num_layers):
        lw = LayerWeights()
        for k, v in _layer(cfg, seed, li).items():
            setattr(lw, k, v)
        model.layers.append(lw)

    seqs = _sequences(case)
    ctx = [c + n for c, n in seqs]
    n_pages = [-(-c // PAGE) for c in ctx]
    width = max(n_pages)
    order = np.random.RandomState(seed & 0x7FFFFFFF).permutation(sum(n_pages))
    pages = np.split(order, np.cumsum(n_pages)[:-1])
    pool = torch.zeros((sum(n_pages), cfg.num_layers, 2, cfg.num_kv_heads, PAGE * cfg.head_dim), dtype=BF16, device=DEV)

    def slots(pg, lo, hi):
        t = np.arange(lo, hi)
        return torch.from_numpy(pg[t // PAGE] * PAGE + t % PAGE).to(DEV)

    for s, ((cached, _), pg) in enumerate(zip(seqs, pages)):
        if cached:
            at, zero = slots(pg, 0, cached), torch.zeros(cached, dtype=torch.int32, device=DEV)
            for li in range(cfg.num_layers):
                ops.kv_cache_write(_history(cfg, seed, li, s, cached), zero, at, model.cos_sin, pool, li, 0,
                                   cfg.num_kv_heads, cfg.head_dim, rotary=False)

    table = _dev([list(map(int, p)) + [0] * (width - len(p)) for p in pages], torch.int32)
    rows = sum(n for _, n in seqs)
    meta = BatchMeta(positions=torch.cat([torch.arange(c, c + n, dtype=torch.int32) for c, n in seqs]).to(DEV),
                     slots=torch.cat([slots(pg, c, c + n) for (c, n), pg in zip(seqs, pages)]))
    ids = _tokens(cfg, seed, rows)
    if case["kind"] == "decode":
        meta.num_decode = rows
        meta.dec_block_tables, meta.dec_ctx_lens = table, _dev(ctx, torch.int32)
        meta.dec_num_splits = ops.decode_num_splits(rows, cfg.num_kv_heads, MAX_LEN)
        shape = (rows, cfg.num_heads, meta.dec_num_splits)
        meta.dec_ws_o = torch.empty((*shape, cfg.head_dim), dtype=torch.float32, device=DEV)
        meta.dec_ws_ml = torch.empty((*shape, 2), dtype=torch.float32, device=DEV)
    else:
        lens = [n for _, n in seqs]
        cu = [0] + list(np.cumsum(lens))
        nq, nkv = cfg.num_heads, cfg.num_kv_heads
        meta.num_prefill_seqs = len(seqs)
        meta.pre_block_tables, meta.pre_ctx_lens = table, _dev(ctx, torch.int32)
        meta.pre_cu_q = _dev([int(c) for c in cu], torch.int32)
        meta.pre_tile_rows = ops.prefill_tile_rows(lens, nq, nkv)
        ts, tq = ops.build_prefill_tiles(lens, nq, nkv, meta.pre_tile_rows, ctx)
        cut = ops.plan_prefill_splits(ts, tq, lens, ctx, nq, nkv, meta.pre_tile_rows)
        if cut is not None:
            ts, tq, split, groups, records = cut
            meta.pre_split, meta.pre_split_groups = _dev(split, torch.int32), _dev(groups, torch.int32)
            meta.pre_split_ws = torch.empty(records * ops.prefill_split_record_bytes(nq, nkv) // 4, dtype=torch.float32, device=DEV)
        meta.pre_tile_seq, meta.pre_tile_q0 = _dev(ts, torch.int32), _dev(tq, torch.int32)
        meta.logits_rows = _dev([int(c) - 1 for c in cu[1:]], torch.int64)
    state = {"model": model, "pool": pool, "meta": meta, "ids": ids}
    if case["kind"] != "prefill":
        state["graph"], state["logits"] = _captured(lambda: model.compute_logits(model.forward(ids, pool, meta)))
    return state


def _prepare_latent(case, seed):
    x = _latent_inputs(case, seed)
    state = {k: x[k] for k in ("q_lat", "q_rot", "pool", "sink")}
    state["pos"], state["table"] = _dev(x["pos"], torch.int32), _dev(x["table"], torch.int32)
    state["seq"] = state["tiles"] = None
    state["splits"] = 1
    if case["mode"] == "decode":
        state["splits"] = ops.decode_num_splits(case["batch"], 1, MAX_LEN)
    else:
        state["seq"] = _dev(x["seq"], torch.int32)
        state["tiles"] = torch.from_numpy(ops.build_latent_tiles([case["batch"]], x["ctx"], case["heads"])).to(DEV)
    return state


def _prepare_scan(case, seed):
    x = _scan_inputs(case, seed)
    lens, h = _scan_lens(case), case["heads"]
    args = {}
    if "decay" in x:
        args = {"decay": _dev(x["decay"], torch.float32), "cos_sin": ops.build_cos_sin(128, MAX_LEN, 10000.0, device=DEV),
                "rot_dims": 128, "layout": 0, "k_scale": 128 ** -0.5, "min_decay": min(x["decay"])}
    else:
        args = {"gate_bias": x["bias"], "gate_lower": x["lower"]}
    cut = ops.build_scan_pieces(lens)
    if cut is not None:
        args["pieces"] = tuple(torch.from_numpy(c).to(DEV) for c in cut)
    return {"proj": x["proj"], "vdim": x["vdim"], "args": args, "heads": h,
            "state": torch.zeros((len(lens), h * 128 * x["vdim"]), dtype=torch.float32, device=DEV),
            "cu": _dev([0] + [int(c) for c in np.cumsum(lens)], torch.int32),
            "slots": torch.arange(len(lens), dtype=torch.int32, device=DEV),
            "pos": torch.cat([torch.arange(n, dtype=torch.int32) for n in lens]).to(DEV)}


def _serde(case):
    cfg = PRESETS[case["model"]]
    return PageSerde(cfg.num_layers, cfg.num_kv_heads, cfg.head_dim, BF16, "cachegen", _levels(case))


@torch.inference_mode()
def prepare(case, seed):
    kind = case["kind"]
    if kind in ("decode", "turn", "prefill"):
        state = _prepare_decoder(case, seed)
    elif kind == "latent":
        state = _prepare_latent(case, seed)
    elif kind == "scan":
        state = _prepare_scan(case, seed)
    elif kind == "speech":
        model = WhisperModel(WHISPER_PRESETS[case["model"]], BF16, DEV)
        model.w = _speech_weights(case, seed)
        state = {"model": model, "mel": _mel(case, seed)}
    else:
        serde = _serde(case)
        pages = [_page(case, seed, i) for i in range(case["pages"])]
        state = {"serde": serde, "pages": pages, "store": [np.zeros(2 * p.numel(), dtype=np.uint8) for p in pages]}
        if kind == "kv_decode":
            state = {"serde": serde, "blobs": [serde.encode(p) for p in pages]}
    state["kind"] = kind
    return state


# ------------------------------------------------------------------------------------------------ one pass
@torch.inference_mode()
def run(state):
    kind = state["kind"]
    if "graph" in state:
        state["graph"].replay()
        return {"logits": state["logits"]}
    if kind == "prefill":
        m = state["model"]
        logits = m.compute_logits(m.forward(state["ids"], state["pool"], state["meta"]))
        return {"logits": logits, "cache": state["pool"]}
    if kind == "latent":
        return ops.latent_attention(state["q_lat"], state["q_rot"], state["pool"], 0, state["table"], state["seq"],
                                    state["pos"], state["sink"], LATENT_SCALE, tiles=state["tiles"], splits=state["splits"])
    if kind == "scan":
        h = state["heads"]
        o = ops.recurrent_scan(state["proj"], 0, h * 128, 2 * h * 128, h, 128, state["vdim"], state["state"], 0, state["cu"],
                               state["slots"], state["pos"], **state["args"])
        return {"out": o, "state": state["state"]}
    if kind == "speech":
        return state["model"].encode(state["mel"])
    if kind == "kv_encode":  # every blob goes into the store's buffer
        for p, to in zip(state["pages"], state["store"]):
            blob = np.frombuffer(state["serde"].encode(p), dtype=np.uint8)
            to[:blob.size] = blob
        return state["store"]
    return [state["serde"].decode(b, DEV) for b in state["blobs"]]


# ------------------------------------------------------------------------------------------------ what a pass cannot do without
def work(case):
    kind = case["kind"]
    if kind in ("decode", "turn", "prefill"):
        cfg = _config(case)
        h, i, v, d = cfg.hidden_size, cfg.intermediate_size, cfg.vocab_size, cfg.head_dim
        nq, nkv = cfg.num_heads, cfg.num_kv_heads
        seqs = _sequences(case)
        rows, outs = sum(n for _, n in seqs), len(seqs)
        attn = h * (nq + 2 * nkv) * d + nq * d * h
        if cfg.num_experts:
            # experts that the step's tokens reach, with even routing
            e, k = cfg.num_experts, cfg.num_experts_per_tok
            held = e * (1 - (1 - k / e) ** rows) * 3 * h * i
            used = k * 3 * h * i
        else:
            held = used = 3 * h * i
        weights = cfg.num_layers * (attn + held) + v * h
        flops = 2 * rows * cfg.num_layers * (attn + used) + 2 * outs * v * h
        cache = 0
        for c, n in seqs:
            cache += (c + n) * 2 * nkv * d  # read once, the new tokens' written
            flops += cfg.num_layers * 4 * nq * d * (n * c + n * (n + 1) // 2)
        return {"bytes": 2 * (weights + cfg.num_layers * cache + rows * h + outs * v), "flops": flops}
    if kind == "latent":
        h, n = case["heads"], case["batch"]
        if case["mode"] == "decode":
            pairs = entries = sum(c + k for c, k in _sequences({"kind": "decode", "batch": n, "context": case["context"]}))
        else:
            entries, pairs = case["context"], n * (case["context"] - n) + n * (n + 1) // 2
        return {"bytes": 2 * (entries * 576 + n * h * (576 + 512)), "flops": 2 * h * pairs * (576 + 512)}
    if kind == "scan":
        h, t, vd = case["heads"], case["rows"], 256 if case["mode"] == "retention" else 128
        # decay, update and read of the state for every token; chunked forms need more, in matrix products
        return {"bytes": t * h * (2 * (256 + vd) + 4 * vd) + 4 * case["seqs"] * h * 128 * vd, "flops": 5 * t * h * 128 * vd}
    if kind == "speech":
        c = WHISPER_PRESETS[case["model"]]
        b, d, t, f = case["windows"], c.d_model, c.max_source_positions, c.encoder_ffn_dim
        params = 3 * d * (c.num_mel_bins + d) + c.encoder_layers * (4 * d * d + 2 * d * f)
        flops = 2 * b * t * (2 * 3 * c.num_mel_bins * d + 3 * d * d + c.encoder_layers * (4 * d * d + 2 * d * f + 2 * t * d))
        return {"bytes": 2 * params + b * t * (2 * 4 * c.num_mel_bins + 2 * d), "flops": flops}
    cfg = PRESETS[case["model"]]
    elems = cfg.num_layers * 2 * cfg.num_kv_heads * PAGE * cfg.head_dim
    return {"bytes": case["pages"] * elems * 2.85, "flops": 0}  # a page of 16-bit values, and about 0.85 bytes a value coded


# ------------------------------------------------------------------------------------------------ the same in 64 bits
def _rope(x, pos, cfg):
    d = cfg.head_dim
    inv = cfg.rope_theta ** -(torch.arange(0, d // 2, dtype=torch.float64, device=DEV) * 2 / d)
    s = cfg.rope_scaling
    if s:  # Llama 3's long-context frequencies
        wave = 2 * math.pi / inv
        orig, lo, hi, f = s["original_max_position_embeddings"], s["low_freq_factor"], s["high_freq_factor"], s["factor"]
        mix = ((orig / wave) - lo) / (hi - lo)
        inv = inv * (mix.clamp(0, 1) + (1 - mix.clamp(0, 1)) / f)
    a = pos.double()[:, None] * inv[None]
    return _turn(x, a.cos()[:, None], a.sin()[:, None])


def _turn(x, c, s):
    a, b = x.chunk(2, dim=-1)
    return torch.cat([a * c - b * s, b * c + a * s], dim=-1)


def _rms(x, w, eps):
    return x / (x.square().mean(-1, keepdim=True) + eps).sqrt() * w.double()


def _attend(q, k, v, first, scale, sink=None):
    """q [n, heads, d], k [m, heads_k, d], v [m, heads_k, dv]: row i sees keys 0 .. first + i."""
    n, hq, d = q.shape
    m, hk, _ = k.shape
    out = torch.empty((n, hq, v.shape[2]), dtype=torch.float64, device=DEV)
    step = max(1, (1 << 28) // (m * (hq // hk)))
    for h in range(hk):
        g = slice(h * (hq // hk), (h + 1) * (hq // hk))
        kh, vh = k[:, h].contiguous(), v[:, h].contiguous()
        for lo in range(0, n, step):
            hi = min(n, lo + step)
            s = (q[lo:hi, g].reshape(-1, d) @ kh.t()).view(hi - lo, -1, m) * scale
            if n > 1:
                last = torch.arange(first + lo, first + hi, device=DEV)
                s.masked_fill_(torch.arange(m, device=DEV)[None, None] > last[:, None, None], float("-inf"))
            if sink is not None:
                s = torch.cat([s, sink[g].double()[None, :, None].expand(hi - lo, -1, 1)], dim=2)
            p = torch.softmax(s, dim=-1)[:, :, :m]
            out[lo:hi, g] = (p.reshape(-1, m) @ vh).view(hi - lo, -1, v.shape[2])
    return out


def _exact_decoder(case, seed):
    cfg = _config(case)
    nq, nkv, d = cfg.num_heads, cfg.num_kv_heads, cfg.head_dim
    seqs = _sequences(case)
    rows = sum(n for _, n in seqs)
    pos = torch.cat([torch.arange(c, c + n) for c, n in seqs]).to(DEV)
    ends = _ends(cfg, seed)
    x = ends["embed"][_tokens(cfg, seed, rows)].double()
    for li in range(cfg.num_layers):
        w = _layer(cfg, seed, li)
        y = _rms(x, w["ln1"], cfg.norm_eps)
        qkv = (y @ w["wqkv"].double().t()).view(rows, nq + 2 * nkv, d)
        q, k, v = _rope(qkv[:, :nq], pos, cfg), _rope(qkv[:, nq:nq + nkv], pos, cfg), qkv[:, nq + nkv:]
        att, at = [], 0
        for s, (c, n) in enumerate(seqs):
            old = _history(cfg, seed, li, s, c).view(c, 2, nkv, d).double()
            att.append(_attend(q[at:at + n], torch.cat([old[:, 0], k[at:at + n]]), torch.cat([old[:, 1], v[at:at + n]]),
                               c, d ** -0.5))
            at += n
        x = x + torch.cat(att).view(rows, nq * d) @ w["wo"].double().t()
        y = _rms(x, w["ln2"], cfg.norm_eps)
        if cfg.num_experts:
            top, ids = (y @ w["router"].double().t()).topk(cfg.num_experts_per_tok, dim=-1)
            p = torch.softmax(top, dim=-1)
            for e in range(cfg.num_experts):
                r, c = (ids == e).nonzero(as_tuple=True)
                if r.numel():
                    g, u = (y[r] @ w["w13"][e].double().t()).chunk(2, dim=-1)
                    x.index_add_(0, r, p[r, c, None] * ((torch.nn.functional.silu(g) * u) @ w["w2"][e].double().t()))
        else:
            g, u = (y @ w["w_gate_up"].double().t()).chunk(2, dim=-1)
            x = x + (torch.nn.functional.silu(g) * u) @ w["w_down"].double().t()
        del w
    last = torch.tensor(np.cumsum([n for _, n in seqs]) - 1, device=DEV)
    logits = _rms(x[last], ends["norm"], cfg.norm_eps) @ ends["lm_head"].double().t()
    return {"logits": logits, "cache": None} if case["kind"] == "prefill" else {"logits": logits}


def _exact_latent(case, seed):
    x = _latent_inputs(case, seed)
    q = torch.cat([x["q_lat"], x["q_rot"]], dim=2).double()
    outs, at = [], 0
    for s, c in enumerate(x["ctx"]):
        n = x["seq"].count(s)
        ent = x["pool"][torch.tensor(x["table"][s][: -(-c // PAGE)], device=DEV)].view(-1, 576)[:c].double()
        outs.append(_attend(q[at:at + n], ent[:, None], ent[:, None, :512], c - n, LATENT_SCALE, x["sink"]))
        at += n
    return torch.cat(outs)


def _exact_scan(case, seed):
    x = _scan_inputs(case, seed)
    h, t, dim, vd = case["heads"], case["rows"], x["dim"], x["vdim"]
    p = x["proj"].double()
    q, k = (p[:, i * h * dim:(i + 1) * h * dim].view(t, h, dim) for i in (0, 1))
    v = p[:, 2 * h * dim:].view(t, h, vd)
    if "decay" in x:
        pos = torch.cat([torch.arange(n) for n in _scan_lens(case)]).to(DEV)
        inv = 10000.0 ** -(torch.arange(0, dim // 2, dtype=torch.float64, device=DEV) * 2 / dim)
        a = (pos.double()[:, None] * inv[None])[:, None]
        q, k = _turn(q, a.cos(), a.sin()), _turn(k, a.cos(), a.sin()) * dim ** -0.5
        # the decays as the program hands them over, in 32 bits
        decay = torch.tensor(x["decay"], dtype=torch.float32, device=DEV).double()[None, :, None].expand(t, h, dim)
    else:
        lo = x["lower"].double().view(1, h, dim)
        decay = lo + (1 - lo) * torch.sigmoid(k + x["bias"].double().view(1, h, dim))
        q, k = torch.nn.functional.silu(q), 1 - decay
    out = torch.empty((t, h, vd), dtype=torch.float64, device=DEV)
    states, row = [], 0
    for n in _scan_lens(case):
        s = torch.zeros((h, dim, vd), dtype=torch.float64, device=DEV)
        for i in range(row, row + n):
            s.mul_(decay[i, :, :, None]).addcmul_(k[i, :, :, None], v[i, :, None, :])
            torch.bmm(q[i, :, None, :], s, out=out[i, :, None, :])
        states.append(s.reshape(-1))
        row += n
    return {"out": out, "state": torch.stack(states)}


def _exact_speech(case, seed):
    c = WHISPER_PRESETS[case["model"]]
    w = {k: t.double() for k, t in _speech_weights(case, seed).items()}
    fn = torch.nn.functional
    outs = []
    for mel in _mel(case, seed).to(BF16).double():  # the network's input is in 16 bits

        def conv(x, name, stride):  # width 3, padding 1: the three taps of every output side by side
            taps = fn.pad(x, (1, 1)).unfold(1, 3, stride).permute(1, 0, 2).reshape(-1, x.shape[0] * 3)
            y = taps @ w[name + ".weight"].reshape(c.d_model, -1).t() + w[name + ".bias"]
            return fn.gelu(y).t()

        def ln(x, name):
            return fn.layer_norm(x, (c.d_model,), w[name + ".weight"], w[name + ".bias"], 1e-5)

        def lin(x, name):
            return fn.linear(x, w[name + ".weight"], w.get(name + ".bias"))

        x = conv(conv(mel, "encoder.conv1", 1), "encoder.conv2", 2).t() + w["encoder.embed_positions.weight"]
        for i in range(c.encoder_layers):
            p = f"encoder.layers.{i}."
            y = ln(x, p + "self_attn_layer_norm")
            q, k, v = (lin(y, p + f"self_attn.{n}_proj").view(-1, c.encoder_heads, 64).transpose(0, 1).contiguous() for n in "qkv")
            a = torch.softmax(torch.bmm(q, k.transpose(1, 2).contiguous()) * 0.125, dim=-1)
            x = x + lin(torch.bmm(a, v).transpose(0, 1).reshape(-1, c.d_model), p + "self_attn.out_proj")
            x = x + lin(fn.gelu(lin(ln(x, p + "final_layer_norm"), p + "fc1")), p + "fc2")
        outs.append(ln(x, "encoder.layer_norm"))
    return torch.stack(outs)


def _exact_kv_decode(case, seed):
    """What the codec's format keeps of a page: whole steps of a group's scale; key groups as steps from the first of 32."""
    cfg = PRESETS[case["model"]]
    lv = torch.tensor(_levels(case), dtype=torch.float32, device=DEV).view(-1, 1, 1, 1)
    outs = []
    for i in range(case["pages"]):
        x = _page(case, seed, i).float().view(cfg.num_layers, 2, -1, 32, 64)

        def steps(g):  # symbols as the 32-bit format rounds them, and the scale
            top = g.abs().amax(-1, keepdim=True)
            scale = torch.where(top > 0, top / lv, torch.ones_like(top))
            return torch.round(g / scale), scale

        k, v = x[:, 0], x[:, 1]
        qa, sa = steps(k[:, :, :1])
        qd, sd = steps(k - qa * sa)
        anchor = qa.double() * sa.double()
        kd = anchor + qd.double() * sd.double()
        kd[:, :, 0] = anchor[:, :, 0]
        qv, sv = steps(v)
        outs.append(torch.stack([kd, qv.double() * sv.double()], dim=1).view(-1))
    return outs


@torch.inference_mode()
def exact(case, seed):
    kind = case["kind"]
    if kind in ("decode", "turn", "prefill"):
        return _exact_decoder(case, seed)
    if kind == "latent":
        return _exact_latent(case, seed)
    if kind == "scan":
        return _exact_scan(case, seed)
    if kind == "speech":
        return _exact_speech(case, seed)
    if kind == "kv_decode":
        return _exact_kv_decode(case, seed)
    return None  # coded bytes have no value in 64 bits: they stay the same


# ------------------------------------------------------------------------------------------------ how far another may be off
def tolerance(case):
    kind = case["kind"]
    if kind in ("decode", "turn", "prefill"):
        return {"rel": 0.03}   # 16-bit activations through the layers: 0.4 to 1 % off the 64-bit result
    if kind == "latent":
        return {"rel": 8e-3}   # 16-bit weights of the values and result: 0.2 %
    if kind == "scan":
        return {"rel": 4e-6}   # 32-bit sums
    if kind == "speech":
        return {"rel": 0.03}   # 16-bit activations through twelve layers: 0.8 %
    return "exact"
