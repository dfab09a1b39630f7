"""Engine ops.  CUDA(HIP)-device tensors run the hand-written gfx950 kernels from
``libvpsa_kernels.so`` (loaded with ctypes and launched on the current torch stream, so
they are capturable into HIP graphs); CPU tensors run the PyTorch definitions in
``reference.py``.  There is no silent GPU fallback: a GPU tensor with the library
missing raises.
"""

from __future__ import annotations

import os

import ctypes
from ctypes import c_float, c_int, c_long, c_void_p

import torch
from torch.autograd import forward_ad

from .. import _native
from . import reference
from .reference import PAGE, build_cos_sin  # noqa: F401

HEAD_DIM_HIP = 128
_lib = None

# Entry points whose launches a step without a graph waits for: with declared arguments a call takes plain numbers (p: address or
# None, l: long, i: int, f: float), and some 25 of them are no 25 objects on the way (Whisper-base, one window, 45
# launches: 709 -> 475 us; latent decode of 32 rows of 1000 entries 26.9 -> 20.1).
_ARGUMENTS = {
    "vpsa_block_gemm": "pll" "ppp" "ppp" "ip" "llp" "lliiiii" "p",
    "vpsa_layernorm": "pppppiilfp",
    "vpsa_dense_attention": "pllppllplliiiifp",
    "vpsa_chunk_scan": "pliiiiiplppippp" "iifippppp" "ippp",
    "vpsa_latent_attention_mfma": "pllpllplpippiippl" "liifiippip",
    "vpsa_page_decode": "ppplliilppip",
}


def _kernels():
    global _lib
    if _lib is None:
        lib = _native.load("vpsa_kernels")
        for name in (
            "vpsa_rmsnorm", "vpsa_rope_cache", "vpsa_kv_cache_write", "vpsa_paged_prefill_rope", "vpsa_prefill_fuses_rope", "vpsa_silu_mul", "vpsa_argmax_bf16",
            "vpsa_paged_prefill", "vpsa_set_prefill_variant", "vpsa_prefill_tile_rows", "vpsa_set_decode_variant", "vpsa_paged_decode", "vpsa_kv_gather_pages",
            "vpsa_kv_scatter_pages", "vpsa_cachegen_encode", "vpsa_cachegen_decode",
            "vpsa_moe_topk_softmax", "vpsa_moe_router", "vpsa_moe_align", "vpsa_moe_permute", "vpsa_moe_combine",
            "vpsa_moe_gemv", "vpsa_moe_mfma", "vpsa_lora_shrink", "vpsa_lora_expand",
            "vpsa_skinny_gemm", "vpsa_hbm_read_probe", "vpsa_set_gemm_variant", "vpsa_stream_gemm",
            "vpsa_stream_gemm_splits", "vpsa_set_stream_targets", "vpsa_rans_encode",
            "vpsa_rans_decode", "vpsa_fetch", "vpsa_copy_parts", "vpsa_page_decode", "vpsa_sample", "vpsa_grouped_gemm", "vpsa_packed_gemm",
            "vpsa_packed_gemm_splits", "vpsa_set_packed_target", "vpsa_dense_decode_attention", "vpsa_dense_attention", "vpsa_dense_attention_cut",
            "vpsa_tile_gemm", "vpsa_tile_gemm_debug", "vpsa_paged_prefill_split",
            "vpsa_embed_scale", "vpsa_add_rmsnorm", "vpsa_rmsnorm_rows", "vpsa_latent_kv_write", "vpsa_rope_pairs",
            "vpsa_latent_attention", "vpsa_sigmoid_gate", "vpsa_relu_sq", "vpsa_glu_clamp", "vpsa_group_topk",
            "vpsa_gather_rows", "vpsa_moe_finish", "vpsa_latent_mfma_supported", "vpsa_latent_mfma_expanded", "vpsa_latent_attention_mfma",
            "vpsa_moe_mfma_act",
            "vpsa_add_dyt", "vpsa_recurrent_scan", "vpsa_chunk_scan", "vpsa_retention_scan", "vpsa_layernorm", "vpsa_mid_gemm", "vpsa_mid_first_chunk", "vpsa_mid_gemm_splits", "vpsa_mid_gemm_norm", "vpsa_mid_gemm_qkv", "vpsa_row_gemm_takes", "vpsa_row_add", "vpsa_row_qkv", "vpsa_mid_unit_factors", "vpsa_block_gemm", "vpsa_block_gemm_shape", "vpsa_head_rms", "vpsa_short_conv_qkv", "vpsa_window_attention",
            "vpsa_mix_heads", "vpsa_xielu", "vpsa_window_mfma_supported", "vpsa_window_attention_mfma", "vpsa_window_tile_slots",
            "vpsa_gated_add_rmsnorm", "vpsa_pool_blocks", "vpsa_diff_heads",
            "vpsa_window_kv_write",
            "vpsa_embed_rmsnorm", "vpsa_depth_mix_rmsnorm", "vpsa_poly_norm", "vpsa_soft_cap", "vpsa_mingru",
        ):
            getattr(lib, name).restype = c_int
        for name in ("vpsa_prefill_split_record_bytes", "vpsa_rans_workspace", "vpsa_rans_decode_workspace",
                     "vpsa_page_workspace"):
            getattr(lib, name).restype = c_long
        kinds = {"p": c_void_p, "l": c_long, "i": c_int, "f": c_float}
        for name, arguments in _ARGUMENTS.items():
            getattr(lib, name).argtypes = [kinds[a] for a in arguments]
        if os.environ.get("VPSA_PREFILL_VARIANT"):  # pin one prefill kernel for A/B runs
            lib.vpsa_set_prefill_variant(c_int(int(os.environ["VPSA_PREFILL_VARIANT"])))
        _lib = lib
    return _lib


def native_loaded() -> bool:
    return _lib is not None


def set_prefill_variant(v: int) -> int:
    """Select the prefill attention kernel (for in-process A/B timing and tests): -1 automatic,
    0 first generation, 1 second generation without wave priorities, 2 second generation,
    3 second generation with head-major tile order, 4 / 5 third generation (64-row tiles, one wave
    per SIMD) in plain / head-major tile order, 6 / 7 the same without the hand-interleaved
    instruction stream.  Returns the previous selection."""
    return int(_kernels().vpsa_set_prefill_variant(c_int(v)))


def set_decode_variant(v: int) -> int:
    """Select the decode attention kernel (-1: automatic by split count, 0: one register set per
    wave, 1: software-pipelined with two register sets, 2: a wave takes both halves of a page;
    3-5: the same three with non-temporal K/V loads, which the automatic choice takes).
    Returns the previous selection."""
    return int(_kernels().vpsa_set_decode_variant(c_int(v)))


_DEVICE: int | None = None


def bind_device(index: int | None) -> None:
    """One process drives one GPU.  The HIP current device is a per-thread setting that starts
    at 0 in every new thread, and both ``torch.cuda.current_stream()`` and the kernel launches
    of the native library follow it: record the process's device here and every launch from
    any thread (engine loop, executor threads) first moves its thread onto that device."""
    global _DEVICE
    _DEVICE = index


def ensure_device() -> None:
    if _DEVICE is not None and torch.cuda.current_device() != _DEVICE:
        torch.cuda.set_device(_DEVICE)


def _raw_stream() -> int:
    ensure_device()
    return torch._C._cuda_getCurrentRawStream(torch._C._cuda_getDevice())


def _stream():
    return c_void_p(_raw_stream())


def _p(t):
    return c_void_p(t.data_ptr()) if t is not None else c_void_p(0)


def _at(t):
    """``_p`` for entry points with declared arguments."""
    return None if t is None else t.data_ptr()


def _check(rc, name):
    if rc != 0:
        raise RuntimeError(f"{name}: unsupported arguments (rc={rc})")


def _bf16_cuda(*ts):
    for t in ts:
        if t is not None and (not t.is_cuda or t.dtype != torch.bfloat16):
            raise TypeError("HIP kernels take bf16 device tensors")


# --------------------------------------------------------------------------- norms
def rms_norm(x, weight, eps, residual=None, out=None):
    """y = rmsnorm(x [+ residual]) * weight.  ``residual`` is updated in place with the sum."""
    if not x.is_cuda:
        y = reference.rms_norm(x, weight, eps, residual)
        if out is not None:
            out.copy_(y)
            return out
        return y
    _bf16_cuda(x, weight, residual)
    hidden = x.shape[-1]
    x2 = x.view(-1, hidden)
    if x2.stride(-1) != 1:
        raise ValueError("rms_norm: last dim must be contiguous")
    if out is None:
        out = torch.empty((x2.shape[0], hidden), dtype=x.dtype, device=x.device)
    if residual is not None and not residual.is_contiguous():
        raise ValueError("rms_norm: residual must be contiguous")
    rc = _kernels().vpsa_rmsnorm(_p(x2), _p(residual), _p(weight), _p(out), c_int(x2.shape[0]),
                                 c_int(hidden), c_long(x2.stride(0)), c_long(out.stride(0)),
                                 c_float(eps), _stream())
    _check(rc, "rms_norm")
    return out.view(x.shape)


def _lies_with(x, t) -> bool:
    """bf16 on the device of ``x``, on 16 bytes."""
    return t.dtype is torch.bfloat16 and t.device == x.device and t.data_ptr() % 16 == 0


def layer_norm(x, weight, bias, eps, residual=None):
    """y = layer norm(x [+ residual]) * weight + bias.  ``residual`` (contiguous) is updated in place with the sum."""
    hidden = x.shape[-1]
    rows_at = x.stride(0) if x.dim() == 2 and x.shape[0] > 1 else hidden
    if (x.is_cuda and 0 < hidden <= 2048 and hidden % 8 == 0 and rows_at % 8 == 0 and weight is not None and bias is not None
            and weight.shape == bias.shape == (hidden,) and weight.is_contiguous() and bias.is_contiguous()
            and (x.is_contiguous() or (x.dim() == 2 and x.stride(1) == 1))
            and not _followed(x, weight, bias, residual)  # (before the addresses, which a function transform's tensors have not)
            and (residual is None or (residual.is_contiguous() and residual.shape == x.shape and _lies_with(x, residual)))
            and _lies_with(x, x) and _lies_with(x, weight) and _lies_with(x, bias)):
        y = torch.empty(x.shape, dtype=x.dtype, device=x.device)
        rc = _kernels().vpsa_layernorm(x.data_ptr(), _at(residual), weight.data_ptr(), bias.data_ptr(), y.data_ptr(), x.numel() // hidden,
                                       hidden, rows_at, eps, _raw_stream())
        _check(rc, "layer_norm")
        return y
    if residual is not None:
        x = residual.add_(x)
    return torch.nn.functional.layer_norm(x, (hidden,), weight, bias, eps)


# --------------------------------------------------------------------------- rope + cache write
def _generic_attention(t, head_dim) -> bool:
    """The HIP attention kernels are built for head_dim 128 (Llama-3, Mixtral); heads of 64
    channels reach them padded (``kv_head_dim``).  Any other head size on a GPU takes the PyTorch
    definitions: correct, slow, announced once, never chosen for a model the kernels cover."""
    global _warned_generic
    if not t.is_cuda:
        return True
    if head_dim == HEAD_DIM_HIP:
        return False
    if not _warned_generic:
        _warned_generic = True
        import logging

        logging.getLogger("vpsa.ops").warning(
            "head_dim %d: attention runs on the generic PyTorch path (the HIP kernels cover head_dim %d)",
            head_dim, HEAD_DIM_HIP)
    return True


_warned_generic = False

# Heads of 64 channels (OPT, GPT-2, Llama-3.2-1B, Qwen2-0.5B) run on the head_dim-128 kernels with
# their channels zero-padded in the KV cache and in Q: zero channels add nothing to QK^T, and the
# padded half of the output is dropped.  Costs twice the KV bytes of those (small) models and buys
# the MFMA kernels and HIP-graph decode instead of per-sequence PyTorch attention.
PAD_HEAD_64 = os.environ.get("VPSA_PAD_HEAD64", "1") != "0"


def kv_head_dim(head_dim: int, device) -> int:
    """Channels per head as stored in the KV pool of a replica on ``device``."""
    if PAD_HEAD_64 and head_dim == 64 and torch.device(device).type == "cuda":
        return HEAD_DIM_HIP
    return head_dim


_pad_cos_sin: dict = {}


class LayerGroupedPool:
    """A paged KV pool cut by layer: ``groups[g]`` is a pool of its own,
    ``[pages][layers / G][K|V][kv_head][64 x d]``, for layers ``g * per`` to ``(g + 1) * per - 1``
    of every page; page ids are shared.  A decode step of one layer then walks an address range
    G times shorter than with all layers in one page: on an MI355X the K/V read rate of the decode
    kernel falls from 6.7 to 6.2-6.4 TB/s once the pages a step touches lie more than about 60 GB
    apart (address translation), which a 250 GB pool of 8 MiB pages always is.  The price: a page
    is G pieces; the lower tiers copy it piece by piece (``page_parts``), replicas that push pages
    to or take pages from other replicas keep whole pages."""

    def __init__(self, groups):
        self.groups = list(groups)
        self.per = self.groups[0].shape[1]
        assert all(g.shape == self.groups[0].shape and g.is_contiguous() for g in self.groups)

    def for_layer(self, layer: int):
        return self.groups[layer // self.per], layer % self.per

    @property
    def shape(self):  # the pool as a whole: [pages][layers][K|V][kv_head][64 x d]
        s = self.groups[0].shape
        return torch.Size((s[0], self.per * len(self.groups), *s[2:]))

    dtype = property(lambda self: self.groups[0].dtype)
    device = property(lambda self: self.groups[0].device)
    is_cuda = property(lambda self: self.groups[0].is_cuda)

    def numel(self) -> int:
        return sum(g.numel() for g in self.groups)

    def element_size(self) -> int:
        return self.groups[0].element_size()

    def page(self, p: int) -> torch.Tensor:
        """A copy of page ``p`` as one tensor [layers][K|V][kv_head][64 x d]."""
        return torch.cat([g[p] for g in self.groups], dim=0)

    def write_page(self, p: int, page: torch.Tensor) -> None:
        for i, g in enumerate(self.groups):
            g[p].copy_(page[i * self.per:(i + 1) * self.per])


# A page as the lower KV tiers see it is the flat [layers][K|V][kv_head][64 x d] array whatever
# the pool's layout: the pieces of a grouped pool, in group order, are exactly that array.
def page_parts(pool, p: int) -> list:
    """The contiguous device pieces of page ``p``, in layer order."""
    if isinstance(pool, LayerGroupedPool):
        return [g[p] for g in pool.groups]
    return [pool[p]]


def page_numel(pool) -> int:
    n = 1
    for d in pool.shape[1:]:
        n *= int(d)
    return n


def page_tensor(pool, p: int) -> torch.Tensor:
    """Page ``p`` as [layers][K|V][kv_head][64 x d]: a view of a whole-page pool, a copy of a grouped one."""
    return pool.page(p) if isinstance(pool, LayerGroupedPool) else pool[p]


def page_read_into(pool, p: int, flat: torch.Tensor, non_blocking: bool = False) -> None:
    """``flat`` (page_numel elements, any device) <- page ``p``."""
    off = 0
    for part in page_parts(pool, p):
        n = part.numel()
        flat[off:off + n].copy_(part.reshape(-1), non_blocking=non_blocking)
        off += n


def page_assign(pool, p: int, flat: torch.Tensor, non_blocking: bool = False) -> None:
    """Page ``p`` <- ``flat`` (page_numel elements, any device)."""
    off = 0
    for part in page_parts(pool, p):
        n = part.numel()
        part.view(-1).copy_(flat[off:off + n], non_blocking=non_blocking)
        off += n


def attention_block(qkv, pool, layer, meta, n_q, n_kv, head_dim, scale, cos_sin, rotary=True):
    """Rotary embedding, KV-cache write and paged attention of one layer for a mixed batch
    (``meta.num_decode`` decode rows first, then the prefill rows).  qkv [T, (n_q + 2 n_kv) * d];
    returns the attention output [T, n_q * d]."""
    if isinstance(pool, LayerGroupedPool):
        pool, layer = pool.for_layer(layer)
    t = qkv.shape[0]
    d = head_dim
    dk = kv_head_dim(d, qkv.device)
    if dk != d:
        # rotate at the true width, then widen every head with zero channels
        if rotary:
            reference.rope_and_cache(qkv, meta.positions, None, cos_sin, pool, layer, n_q, n_kv, d, True)
        wide = torch.nn.functional.pad(qkv.view(t, n_q + 2 * n_kv, d), (0, dk - d)).view(t, -1)
        cs = _pad_cos_sin.get(qkv.device)
        if cs is None:
            cs = _pad_cos_sin[qkv.device] = torch.zeros((1, dk), dtype=torch.float32, device=qkv.device)
        out = _attention_block(wide, pool, layer, meta, n_q, n_kv, dk, scale, cs, False)
        return out.view(t, n_q, dk)[:, :, :d].reshape(t, n_q * d)
    return _attention_block(qkv, pool, layer, meta, n_q, n_kv, d, scale, cos_sin, rotary)


def prefill_fuses_rope(n_q: int, n_kv: int, tile_rows) -> bool:
    """True when the prefill kernel that will run rotates its query rows itself."""
    return bool(tile_rows) and int(_kernels().vpsa_prefill_fuses_rope(c_int(n_q), c_int(n_kv), c_int(tile_rows))) == 1


def _attention_block(qkv, pool, layer, meta, n_q, n_kv, d, scale, cos_sin, rotary):
    nd = meta.num_decode
    # Prefill rows: their K / V go to the cache through the tile kernel (rotated K, V transposed
    # in LDS so that the page's [channel][32 keys] runs are written whole), and the query rows are
    # rotated by the attention kernel as it loads them when the kernel that will run can do that
    # (GQA groups of 4 and multiples), else in place by a pass over the query heads only.  Decode
    # rows keep the per-token pass with the in-place rotation: their kernel reads q as stored.
    tiled = meta.num_prefill_seqs > 0 and not _generic_attention(qkv, d)
    fuse = tiled and rotary and prefill_fuses_rope(n_q, n_kv, meta.pre_tile_rows)
    if tiled:
        if nd > 0:
            rope_and_cache(qkv[:nd], meta.positions[:nd], meta.slots[:nd], cos_sin, pool, layer, n_q, n_kv, d,
                           rotary)
        kv_cache_write(qkv[nd:], meta.positions[nd:], meta.slots[nd:], cos_sin, pool, layer, n_q, n_kv, d,
                       rotary)
        if rotary and not fuse:
            rope_and_cache(qkv[nd:], meta.positions[nd:], None, cos_sin, pool, layer, n_q, 0, d, True)
    else:
        rope_and_cache(qkv, meta.positions, meta.slots, cos_sin, pool, layer, n_q, n_kv, d, rotary)
    t = qkv.shape[0]
    alloc = torch.zeros if getattr(meta, "pre_padded", False) else torch.empty
    out = alloc((t, n_q * d), dtype=qkv.dtype, device=qkv.device)
    q = qkv[:, : n_q * d]
    if nd > 0:
        paged_decode(q[:nd], out[:nd], pool, layer, meta.dec_block_tables, meta.dec_ctx_lens, n_q, n_kv, d,
                     scale, getattr(meta, "dec_num_splits", 1) or 1, getattr(meta, "dec_ws_o", None),
                     getattr(meta, "dec_ws_ml", None))
    if meta.num_prefill_seqs > 0:
        paged_prefill(q[nd:], out[nd:], pool, layer, meta.pre_block_tables, meta.pre_cu_q, meta.pre_ctx_lens,
                      meta.pre_tile_seq, meta.pre_tile_q0, n_q, n_kv, d, scale, meta.pre_tile_rows,
                      rope=cos_sin if fuse else None, split=getattr(meta, "pre_split", None),
                      split_ws=getattr(meta, "pre_split_ws", None), groups=getattr(meta, "pre_split_groups", None))
    return out


def kv_cache_write(qkv, positions, slots, cos_sin, pool, layer, n_q, n_kv, head_dim, rotary=True):
    """K (rotated) and V heads of ``qkv`` rows -> paged cache; ``qkv`` itself is not modified and
    the query heads are not read (prefill rows: their queries are rotated by ``paged_prefill(rope=)``
    or by a query-only ``rope_and_cache`` pass).  ``rotary=False`` writes K as it is."""
    _bf16_cuda(qkv, pool)
    assert positions.dtype == torch.int32 and slots.dtype == torch.int64
    assert cos_sin.dtype == torch.float32 and cos_sin.shape[1] == head_dim == 128
    base = pool.data_ptr() + layer * pool.stride(1) * 2
    rc = _kernels().vpsa_kv_cache_write(_p(qkv), _p(positions), _p(slots), _p(cos_sin), c_void_p(base),
                                        c_int(qkv.shape[0]), c_long(qkv.stride(0)), c_int(n_q),
                                        c_int(n_kv), c_long(pool.stride(0)), c_long(pool.stride(2)),
                                        c_int(1 if rotary else 0), _stream())
    _check(rc, "kv_cache_write")


def rope_and_cache(qkv, positions, slots, cos_sin, pool, layer, n_q, n_kv, head_dim, rotary=True):
    if _generic_attention(qkv, head_dim):
        return reference.rope_and_cache(qkv, positions, slots, cos_sin, pool, layer, n_q, n_kv,
                                        head_dim, rotary)
    _bf16_cuda(qkv, pool)
    assert positions.dtype == torch.int32 and (slots is None or slots.dtype == torch.int64)
    assert cos_sin.dtype == torch.float32 and cos_sin.shape[1] == head_dim
    base = pool.data_ptr() + layer * pool.stride(1) * 2
    rc = _kernels().vpsa_rope_cache(_p(qkv), _p(positions), _p(slots), _p(cos_sin), c_void_p(base),
                                    c_int(qkv.shape[0]), c_long(qkv.stride(0)), c_int(n_q),
                                    c_int(n_kv), c_long(pool.stride(0)), c_long(pool.stride(2)),
                                    c_int(1 if rotary else 0), _stream())
    _check(rc, "rope_and_cache")


# --------------------------------------------------------------------------- attention
def prefill_tile_rows(q_lens, n_q, n_kv) -> int:
    """Query rows per work-list entry.  The third-generation kernel works on 64-row tiles (one
    GQA group of 4 heads x 64 rows per workgroup) and is taken whenever the GQA ratio is a
    multiple of 4.  The choice deliberately does not look at the batch: two kernels round
    differently, and a request's tokens must not depend on what shares its step."""
    del q_lens
    rows = int(_kernels().vpsa_prefill_tile_rows(c_int(n_q), c_int(n_kv), c_int(1)))
    if rows <= 0:
        raise ValueError(f"paged_prefill: unsupported head layout n_q={n_q} n_kv={n_kv}")
    return rows


def build_prefill_tiles(q_lens, n_q, n_kv, rows=None, ctx_lens=None):
    """Host-side work list for the prefill kernel: one (sequence, first row) entry per query
    tile of ``rows`` rows (default: ``prefill_tile_rows``).  Sequences with the longest context
    come first (the heaviest workgroups start earliest) and a sequence's tiles stay together,
    longest first: the workgroups that run side by side on one XCD then stream the SAME K/V
    pages through its L2 instead of one stream per sequence (8 equal sequences interleaved cost
    the kernel a fifth of its throughput in HBM waits)."""
    qt = rows or prefill_tile_rows(q_lens, n_q, n_kv)
    weight = ctx_lens if ctx_lens is not None else q_lens
    seqs, q0s = [], []
    for s in sorted(range(len(q_lens)), key=lambda i: -weight[i]):
        for q0 in range((q_lens[s] - 1) // qt * qt, -1, -qt):
            seqs.append(s)
            q0s.append(q0)
    return seqs, q0s


# Work lists that leave the chip part-filled are cut along the key range: one new turn behind a
# 21k-token history is 8 workgroups that each walk 330 key tiles alone (10 ms on a 256-CU chip), and
# 288 equal workgroups run as one full round and a nearly empty second.  The pieces run as
# workgroups of their own and leave partials for a merge pass.  One workgroup occupies a CU (96 KiB
# of LDS), so plans are priced in rounds of TILE_CUS workgroups.
SPLIT_MIN_KEY_TILES = 8     # a piece is at least this long (the kernel needs >= 3 in the last one)
SPLIT_MAX_ROUNDS = 3        # longer lists lose at most a quarter of a round and are left alone
SPLIT_CANDIDATES = 8        # round counts tried, starting at the list's own
SPLIT_WG_OVERHEAD = 7.0     # a workgroup's prologue + epilogue, in key-tile times (1.9 us; a lone round of n tiles takes 14 + 1.9 n)
SPLIT_MERGE_COST = 6.0      # the merge launch, in key-tile times (7 to 8 us and the gap before it; at 25, the times before the stroke: 16 rows
                            # behind 2000 tokens 50/22 us, 97 behind 2000 56/28, 512 behind 2000 66/43, 2900 behind 12000 642/590)
SPLIT_RECORD_COST = 0.15    # writing + reading one partial record, in key-tile times
PREFILL_SPLITS = os.environ.get("VPSA_PREFILL_SPLITS", "1") != "0"


def prefill_split_record_bytes(n_q: int, n_kv: int) -> int:
    return int(_kernels().vpsa_prefill_split_record_bytes(c_int(n_q), c_int(n_kv)))


def prefill_splits_supported(n_q: int, n_kv: int, rows: int) -> bool:
    """Only the 64-row kernel (GQA ratios of 3 and up: workgroups of 4 heads, the last one of a KV
    head padded with spare waves) takes split work lists."""
    return PREFILL_SPLITS and rows == 64 and n_kv > 0 and n_q % n_kv == 0 and n_q // n_kv >= 3


def _whole_cost(kts, head_groups):
    """Modelled time of the uncut list in key-tile times.  Workgroups start longest first, so the
    chip stays full until the last, partial round, which is made of the shortest entries."""
    total = sum(kts) + SPLIT_WG_OVERHEAD * len(kts)
    wgs = len(kts) * head_groups
    tail = (TILE_CUS - wgs % TILE_CUS) % TILE_CUS / TILE_CUS * (min(kts) + SPLIT_WG_OVERHEAD)
    return max(max(kts) + SPLIT_WG_OVERHEAD, total * head_groups / TILE_CUS + tail)


def _split_counts(lengths, budget):
    """``lengths``: {key tiles: entries of that length}.  Pieces per entry of each length so that
    the longest piece is as short as ``budget`` entries in all allow; None when the budget does not
    cover the list."""
    def entries(piece):
        return sum(m * max(1, min(-(-kt // piece), kt // SPLIT_MIN_KEY_TILES)) for kt, m in lengths.items())
    lo, hi = SPLIT_MIN_KEY_TILES, max(lengths)
    if entries(hi) > budget:
        return None
    while lo < hi:
        mid = (lo + hi) // 2
        if entries(mid) <= budget:
            hi = mid
        else:
            lo = mid + 1
    return {kt: max(1, min(-(-kt // lo), kt // SPLIT_MIN_KEY_TILES)) for kt in lengths}


def plan_prefill_splits(seqs, q0s, q_lens, ctx_lens, n_q, n_kv, rows, max_entries=None, max_records=None):
    """Cut the key ranges of a work list that would leave the chip part-filled.  Returns None when
    nothing is to be split, else (seqs, q0s, split, groups, n_records): the expanded work list,
    ``split`` = 3 ints per entry (first key tile, end key tile, partial record or -1), ``groups`` =
    4 ints per split tile (sequence, first row, first record, records).

    The uncut list is priced with the chip kept full (what longest-first dispatch achieves), a plan
    as whole rounds of its longest piece: a cut has to win against the better case of leaving the
    list alone."""
    if not prefill_splits_supported(n_q, n_kv, rows) or not seqs:
        return None
    head_groups = n_kv * ((n_q // n_kv + 3) // 4)
    if len(seqs) * head_groups > SPLIT_MAX_ROUNDS * TILE_CUS:
        return None
    kts = []
    for s, q0 in zip(seqs, q0s):
        last_row = min(q0 + rows - 1, q_lens[s] - 1)
        kts.append((ctx_lens[s] - q_lens[s] + last_row) // PAGE + 1)
    if max(kts) < 2 * SPLIT_MIN_KEY_TILES:
        return None
    whole = _whole_cost(kts, head_groups)
    ideal = (sum(kts) + SPLIT_WG_OVERHEAD * len(kts)) * head_groups / TILE_CUS
    if whole < 1.1 * ideal + SPLIT_MERGE_COST:  # balanced as it is
        return None
    lengths = {}
    for kt in kts:
        lengths[kt] = lengths.get(kt, 0) + 1
    per_round = max(1, TILE_CUS // head_groups)  # work-list entries that fill the chip once
    first = -(-len(seqs) // per_round)
    best, best_cost = None, 0.95 * whole  # a cut has to pay for itself
    for rounds in range(first, first + (SPLIT_CANDIDATES if len(lengths) <= 16 else 3)):
        budget = rounds * per_round
        if max_entries is not None:
            budget = min(budget, max_entries)
        if max_records is not None:  # every entry may end up with a record of its own
            budget = min(budget, max_records)
        counts = _split_counts(lengths, budget)
        if counts is None or max(counts.values()) == 1:
            continue
        n = sum(m * counts[kt] for kt, m in lengths.items())
        records = sum(m * counts[kt] for kt, m in lengths.items() if counts[kt] > 1)
        longest = max(-(-kt // c) for kt, c in counts.items())
        cost = (-(-n * head_groups // TILE_CUS) * (longest + SPLIT_WG_OVERHEAD)
                + SPLIT_MERGE_COST + SPLIT_RECORD_COST * records * head_groups / 8)
        if cost < best_cost:
            best, best_cost = counts, cost
    if best is None:
        return None
    best = [best[kt] for kt in kts]
    seqs2, q0s2, split, groups = [], [], [], []
    rec = 0
    for s, q0, kt, c in zip(seqs, q0s, kts, best):
        if c == 1:
            seqs2.append(s)
            q0s2.append(q0)
            split += [0, kt, -1]
            continue
        groups += [s, q0, rec, c]
        base, extra = divmod(kt, c)
        k0 = 0
        for j in range(c):
            k1 = k0 + base + (1 if j < extra else 0)
            seqs2.append(s)
            q0s2.append(q0)
            split += [k0, k1, rec]
            rec += 1
            k0 = k1
    return seqs2, q0s2, split, groups, rec


def paged_prefill(q, out, pool, layer, block_tables, cu_q, ctx_lens, tile_seq, tile_q0, n_q, n_kv,
                  head_dim, scale, tile_rows=None, rope=None, split=None, split_ws=None, groups=None):
    """``tile_rows``: the tile height ``tile_seq`` / ``tile_q0`` were built for (default: the
    32-row-wave layout of the first two kernel generations).  ``rope``: the [position, head_dim]
    fp32 cos / sin table when ``q`` holds unrotated rows (``prefill_fuses_rope`` says whether the
    kernel that will run takes it)."""
    if _generic_attention(q, head_dim):
        return reference.paged_prefill(q, out, pool, layer, block_tables, cu_q, ctx_lens, n_q,
                                       n_kv, head_dim, scale)
    _bf16_cuda(q, out, pool)
    for t in (block_tables, cu_q, ctx_lens, tile_seq, tile_q0):
        assert t.dtype == torch.int32 and t.is_cuda and t.is_contiguous()
    assert tile_seq.numel() == tile_q0.numel()
    assert cu_q.numel() == ctx_lens.numel() + 1 and block_tables.shape[0] >= ctx_lens.numel()
    if tile_rows is None:
        tile_rows = 32 * (4 // min(n_q // n_kv, 4))
    base = pool.data_ptr() + layer * pool.stride(1) * 2
    assert rope is None or (rope.dtype == torch.float32 and rope.is_contiguous() and rope.shape[1] == head_dim)
    if split is not None:
        # split [entries][3], groups [n][4] (int32 on the device), split_ws fp32 with room for every record
        assert split.dtype == torch.int32 and split.numel() == 3 * tile_seq.numel() and split.is_contiguous()
        assert groups.dtype == torch.int32 and groups.numel() % 4 == 0 and groups.is_contiguous()
        assert split_ws.dtype == torch.float32 and split_ws.is_contiguous()
    rc = _kernels().vpsa_paged_prefill_split(
        _p(q), c_long(q.stride(0)), _p(out), c_long(out.stride(0)), c_void_p(base),
        c_long(pool.stride(0)), c_long(pool.stride(2)), _p(block_tables),
        c_int(block_tables.stride(0)), _p(cu_q), _p(ctx_lens), _p(tile_seq), _p(tile_q0),
        c_int(tile_seq.numel()), c_int(ctx_lens.numel()), c_int(tile_rows), c_int(n_q), c_int(n_kv),
        c_float(scale), _p(rope), _p(split), _p(split_ws), _p(groups),
        c_int(0 if groups is None else groups.numel() // 4), _stream())
    _check(rc, "paged_prefill")


def dense_decode_attention_supported(q, k, v, heads: int) -> bool:
    """Shapes the dense single-query kernel covers: bf16 on the GPU, 64-channel heads, unit
    stride over channels, 16-byte aligned rows."""
    d = q.shape[-1]
    if not all(t.is_cuda and t.dtype == torch.bfloat16 for t in (q, k, v)):
        return False
    return (d == heads * 64 and q.dim() == 2 and k.dim() == 3
            and k.shape == v.shape and k.stride() == v.stride() and k.shape[0] == q.shape[0] and k.shape[2] == d
            and q.stride(1) == 1 and k.stride(2) == 1 and q.stride(0) % 8 == 0 and k.stride(0) % 8 == 0
            and k.stride(1) % 8 == 0 and (q.data_ptr() | k.data_ptr() | v.data_ptr()) % 16 == 0)


def dense_decode_attention(q, k, v, heads: int, pos=None, out=None):
    """softmax(q k^T / 8) v for ONE query per batch row over dense K/V: q [B, heads * 64],
    k / v [B, T, heads * 64] -> [B, heads * 64].  ``pos`` (one int64 on the device) limits the
    keys to positions 0..pos; None attends to all T.  Graph-capturable."""
    b, d = q.shape
    if out is None:
        out = torch.empty((b, d), dtype=q.dtype, device=q.device)
    rc = _kernels().vpsa_dense_decode_attention(
        _p(q), c_long(q.stride(0)), _p(k), _p(v), c_long(k.stride(0)), c_long(k.stride(1)), _p(pos),
        c_int(b), c_int(heads), c_int(k.shape[1]), _p(out), c_long(out.stride(0)), c_float(0.125), _stream())
    _check(rc, "dense_decode_attention")
    return out


def dense_attention_supported(q, k, v, heads: int) -> bool:
    """Shapes the dense bidirectional kernel covers: bf16 on the GPU, [B, T, heads * 64] with unit
    stride over channels and 16-byte aligned rows."""
    for t in (q, k, v):
        if not t.is_cuda or t.dtype is not torch.bfloat16 or t.dim() != 3:
            return False
    d, ks, qst, kst = q.shape[-1], k.shape, q.stride(), k.stride()
    return (d == heads * 64 and ks == v.shape and kst == v.stride() and ks[0] == q.shape[0]
            and ks[2] == d and ks[1] > 0 and qst[2] == 1 and kst[2] == 1
            and (qst[0] | qst[1] | kst[0] | kst[1]) % 8 == 0
            and (q.data_ptr() | k.data_ptr() | v.data_ptr()) % 16 == 0)


def dense_attention(q, k, v, heads: int, out=None):
    """softmax(q k^T / 8) v with every query attending to every key: q [B, Tq, heads * 64],
    k / v [B, Tk, heads * 64] -> [B, Tq, heads * 64] (MFMA flash kernel, scores never stored)."""
    b, tq, d = q.shape
    if out is None:
        out = torch.empty((b, tq, d), dtype=q.dtype, device=q.device)
    qs, ks, os_ = q.stride(), k.stride(), out.stride()
    rc = _kernels().vpsa_dense_attention(q.data_ptr(), qs[0], qs[1], k.data_ptr(), v.data_ptr(), ks[0], ks[1], out.data_ptr(), os_[0], os_[1],
                                         b, heads, tq, k.shape[1], 0.125, _raw_stream())
    _check(rc, "dense_attention")
    return out


def decode_num_splits(num_seqs: int, n_kv: int, max_ctx: int) -> int:
    """Splits of the key range per (sequence, KV head).  Measured on 21.5k-token contexts in the
    engine's page layout with streaming loads (`benchmarks/attn_micro.py --cases decode --layers 32
    --decode-seqs 4,8,16,24,40,64`): batches of a few sequences read fastest with about one
    workgroup per CU (4 sequences: 5.25 TB/s at 192 workgroups, 4.7 at 1024), larger ones with about
    three (16 sequences: 6.5-6.6 TB/s at 512-768 workgroups, 40 sequences: 6.45 at 960, 6.35 at
    640 or 1280); at least 256 keys per split."""
    per_split = max(1, num_seqs * n_kv)
    target = 256 if per_split < 96 else 768
    want = max(1, -(-target // per_split))
    by_len = max(1, max_ctx // 256)
    return int(max(1, min(want, by_len, 32)))


def paged_decode(q, out, pool, layer, block_tables, ctx_lens, n_q, n_kv, head_dim, scale,
                 num_splits=1, ws_o=None, ws_ml=None):
    if _generic_attention(q, head_dim):
        return reference.paged_decode(q, out, pool, layer, block_tables, ctx_lens, n_q, n_kv,
                                      head_dim, scale)
    _bf16_cuda(q, out, pool)
    assert block_tables.dtype == torch.int32 and ctx_lens.dtype == torch.int32
    n = q.shape[0]
    assert block_tables.shape[0] >= n and ctx_lens.numel() >= n
    if num_splits > 1:
        if ws_o is None:
            ws_o = torch.empty((n, n_q, num_splits, head_dim), dtype=torch.float32, device=q.device)
            ws_ml = torch.empty((n, n_q, num_splits, 2), dtype=torch.float32, device=q.device)
        assert ws_o.numel() >= n * n_q * num_splits * head_dim
    base = pool.data_ptr() + layer * pool.stride(1) * 2
    rc = _kernels().vpsa_paged_decode(
        _p(q), c_long(q.stride(0)), _p(out), c_long(out.stride(0)), c_void_p(base),
        c_long(pool.stride(0)), c_long(pool.stride(2)), _p(block_tables),
        c_int(block_tables.stride(0)), _p(ctx_lens), _p(ws_o), _p(ws_ml), c_int(n), c_int(n_q),
        c_int(n_kv), c_int(num_splits), c_float(scale), _stream())
    _check(rc, "paged_decode")


# --------------------------------------------------------------------------- projections
SKINNY_MAX_ROWS = 64
_skinny_enabled = os.environ.get("VPSA_SKINNY_GEMM", "1") != "0"


def set_skinny_gemm(on: bool) -> bool:
    """Switch the decode-batch projection kernels on or off (A/B timing); returns the old value."""
    global _skinny_enabled
    old, _skinny_enabled = _skinny_enabled, bool(on)
    return old


def set_gemm_variant(v: int) -> int:
    """Tiling knobs of the decode-batch projection kernel (bit 0: eight loads per operand in
    flight instead of four, bit 1: four waves per workgroup); returns the previous value."""
    return int(_kernels().vpsa_set_gemm_variant(c_int(v)))


def _skinny(x2, w, bias, pair):
    n_out = w.shape[0] // 2 if pair else w.shape[0]
    out = torch.empty((x2.shape[0], n_out), dtype=x2.dtype, device=x2.device)
    rc = _kernels().vpsa_skinny_gemm(_p(x2), c_long(x2.stride(0)), _p(w), _p(bias), _p(out),
                                     c_long(out.stride(0)), c_int(x2.shape[0]), c_int(w.shape[0]),
                                     c_int(w.shape[1]), c_int(1 if pair else 0), _stream())
    return out if rc == 0 else None


def _stream_gemm(x2, w, bias, pair):
    """Streaming projection kernel (LDS-staged, reduction split across workgroups)."""
    lib = _kernels()
    m, n, k = x2.shape[0], w.shape[0], w.shape[1]
    splits = int(lib.vpsa_stream_gemm_splits(c_int(m), c_int(n), c_int(k), c_int(1 if pair else 0)))
    if splits <= 0:
        return None
    out = torch.empty((m, n // 2 if pair else n), dtype=x2.dtype, device=x2.device)
    ws = torch.empty((splits * m * n,), dtype=torch.float32, device=x2.device) if splits > 1 else None
    rc = lib.vpsa_stream_gemm(_p(x2), c_long(x2.stride(0)), _p(w), _p(bias), _p(out), c_long(out.stride(0)),
                              _p(ws), c_int(m), c_int(n), c_int(k), c_int(1 if pair else 0),
                              c_int(splits), _stream())
    return out if rc == 0 else None


# ``mid_gemm`` (128 weight rows a workgroup, both operands straight into LDS) against what ran before, microseconds in a graph over
# weights that no cache holds (library with its activation pass, or the kernels above up to 16 rows / mid_gemm):
#   28672 x 4096 pair    1 row 43.6/36.6    24 rows 51.1/36.6    64 rows 51.7/38.5    112 rows 56.8/48.2    128 rows 56.3/50.7
#   4096 x 14336         1     25.1/22.4    24      27.5/23.7    64      38.6/27.9    128      71.2/35.7    200      54.1/48.2
#   6144 x 4096          1     12.9/12.5    24      15.1/14.2    64      18.3/17.0    112      23.9/20.6    200      26.1/30.6
#   4096 x 4096          1      9.8/9.7     24      13.4/11.5    64      15.2/13.4     97      16.3/16.4
#   128256 x 4096        1      190/160     24       196/164     64       208/183     112       232/213     128       233/224
#   57344 x 8192 pair    1      172/146     64       194/150     112      200/178     128       203/186     160       208/364
#   28672 x 8192 pair    1      113/72      64       101/72      112      111/89      128       112/93      160       121/185
#   8192 x 28672         1       86/71      64       140/89      128      201/112     200      307/172
#   3584 x 18944         1       46/26      24       107/27      64        90/32      128       99/40       200      122/61
#   37888 x 3584 pair    1     48.4/54.1    64      64.8/64.8  (296 workgroups: a second round nearly empty)
#   2048 x 2048          1      5.7/7.4     64       8.7/10.6  (64 workgroups)
MID_MIN_FILL = 0.75      # of the rounds of one workgroup per CU
MID_MIN_FILL_ROWS = 192  # the same as workgroups
MID_ROWS = 96            # every shape that fills the chip
MID_ROWS_BLOCK = 128     # one round or full ones (448 workgroups win by 2 to 6 %), and partial sums (32 bits, written and read) below
MID_BLOCK_FILL = 0.875   # MID_SUMS quarters of the weights' bytes
MID_SUMS = 3
MID_SUMS_NORM = 4        # where the reduction also makes the residual stream and the norm, whose own pass takes 4.9 us beside the library
                         # (with it / mid_gemm, 4096 x 4096: 97 rows 20.2/18.1, 113 21.2/19.7, 128 28.8/20.3; 3584 x 3584: 97 rows 22.4/17.1)
MID_ROWS_LONG = 256      # reductions beyond 8192, where the library's pick is poor at every batch


def _mid_splits(m: int, n: int, k: int, pair: bool, sums: int = MID_SUMS, rows: int = MID_ROWS_BLOCK) -> int:
    """Workgroups along the reduction when ``mid_gemm`` should take the shape, else 0.  ``sums``: quarters of the weights' bytes that
    the partial sums of up to ``rows`` rows may have."""
    if not 0 < m <= MID_ROWS_LONG:
        return 0
    splits = int(_kernels().vpsa_mid_gemm_splits(c_int(m), c_int(n), c_int(k), c_int(1 if pair else 0)))
    if splits <= 0:
        return 0
    wgs = (n // 128) * splits * (-(-m // 128))  # (a pair's workgroup holds 64 gate and 64 up rows)
    if wgs < MID_MIN_FILL * TILE_CUS * (-(-wgs // TILE_CUS)):
        return 0
    if m <= MID_ROWS or (not pair and k > STREAM_MAX_K):
        return splits
    if (m <= rows and (wgs <= TILE_CUS or wgs >= MID_BLOCK_FILL * TILE_CUS * (-(-wgs // TILE_CUS)))
            and (splits == 1 if pair else 16 * m * splits <= sums * k)):
        return splits
    return 0


def _followed(*ts) -> bool:
    """True where something follows a call from outside and would lose sight of it in a kernel launch: gradients of its operands,
    forward-mode tangents, a function transform (vmap), a trace or a dispatch mode."""
    return ((torch.is_grad_enabled() and any(t is not None and t.requires_grad for t in ts)) or forward_ad._current_level >= 0
            or torch._C._functorch.peek_interpreter_stack() is not None or torch._C._get_tracing_state() is not None
            or torch._C._len_torch_dispatch_stack() > 0)


# ``block_gemm``'s projections (one row tile of up to 256 rows or two, split sums closed by mid_gemm's reductions), library with its
# activation or norm pass / mid_gemm / block, the same way:
#   28672 x 4096 pair    97 rows 59.2/47.5/44.8    128 rows 60.2/49.1/48.3    129 rows 61.6/-/49.3    200 rows 71.2/-/55.0    256 rows 72.0/-/58.3
#   57344 x 8192 pair    97      196/198/171       128      196/188/182       129      204/-/187      200      220/-/207      256      221/-/232
#   128256 x 4096        97      233/218/209       128      235/227/219       129      288/-/225      200      297/-/243      256      299/-/264
#   152064 x 3584        97      237/235/241       128      243/250/251       129      257/-/253      200      324/-/273      256      319/-/286
#   4096 x 14336, norm   97      53.8/35.0/35.3    128      80.0/38.3/38.8    129      58.4/46.6/38.1 256      65.8/51.1/45.7 512      93.1/-/68.2
#   8192 x 28672, norm   97      201/107/97        128      211/115/103       129      305/175/104    256      323/172/124    512      314/-/227
#   3584 x 18944, norm   97      97.5/39.2/38.1    128      100/43.2/41.2     129      104/60.3/41.5  256      126/62.6/48.5  512      201/-/82
#   8192 x 8192, norm    97      43.7/36.6/37.4    128      53.9/40.0/39.9    129      52.9/54.5/40.3 256      81.4/57.0/47.8 512      80.9/-/76.7
#   4096 x 4096, norm   129      25.9/21.7/21.9    200      26.2/22.4/23.9    256      26.9/24.2/27.6 300      29.5/-/29.7    512      33.9/-/35.0
#   3584 x 3584, norm   129      23.7/20.3/22.1    200      23.9/21.2/26.0    256      24.5/22.6/27.9 300      27.8/-/28.6    512      30.5/-/32.2
#   6144 x 4096         129      38.4/29.7/24.9    150      39.4/30.4/26.3    176      25.7/30.1/27.3 230      26.3/30.8/29.9 256      39.9/31.6/30.9
#   10240 x 8192        129      58.3/81.1/45.3    200      67.6/82.3/49.4    256      89.1/84.1/54.3 300      75.0/-/88.5    (two row tiles, 160 workgroups)
BLOCK_MIN_ROWS = 97
BLOCK_MAX_ROWS = 256             # one row tile
BLOCK_MAX_ROWS_LONG = 512        # two: split products (unsplit 28672 x 4096, 300 rows: 80 with the library, 104)
BLOCK_MID_ELEMS = 1 << 26        # up to 128 rows mid_gemm keeps split products of smaller weights
BLOCK_SUMS_QKV = 8               # where the reduction also rotates and writes the cache, a launch of 12 us of its own with 256 rows


def _block_splits(m: int, n: int, k: int, pair: bool, sums: int = MID_SUMS) -> int:
    """Workgroups along the reduction when ``block_gemm``'s projections should take the shape, else 0.  ``sums``: quarters of the
    weights' bytes that the partial sums may have (twice their rows: written and read)."""
    if not BLOCK_MIN_ROWS <= m <= BLOCK_MAX_ROWS_LONG:
        return 0
    splits = int(_kernels().vpsa_block_proj_splits(c_int(m), c_int(n), c_int(k), c_int(1 if pair else 0)))
    wgs = -(-n // 128) * splits * (-(-m // BLOCK_MAX_ROWS))
    rounds = -(-wgs // TILE_CUS)
    if splits <= 0 or wgs < (MID_MIN_FILL if rounds == 1 else MID_BLOCK_FILL) * TILE_CUS * rounds:
        return 0
    if splits == 1:
        # In one round always.  In several, each begins and ends once more: up to 128 rows reductions of 64 chunks and more carry that
        # (128256 x 4096, 97 rows 209 us against 218 and 233), of 56 no more (152064 x 3584 241 against 235 and 237; nothing measured between);
        # beyond, the products do, up to 224 rows in any rounds that got here (57344 x 8192, 448 workgroups of 512, 200 rows 207
        # against 220), with rows that fill the tile where the last round is nearly full (256 rows: 152064 x 3584, 1188 of 1280, 286 against 319;
        # 448 of 512, 232 against 221: the line between 0.875 and 0.93).
        if m > BLOCK_MAX_ROWS or (rounds > 1 and (k < STREAM_MAX_K // 2 if m <= MID_ROWS_BLOCK else m > 224 and wgs < 0.9 * TILE_CUS * rounds)):
            return 0
        return splits
    if pair or (m <= MID_ROWS_BLOCK and n * k <= BLOCK_MID_ELEMS) or 16 * m * splits > sums * k:
        return 0
    return splits


def _reads(x2, w, bias) -> bool:
    """Operands that the projection kernels of small batches read."""
    return (_skinny_enabled and x2.is_cuda and w.device == x2.device and x2.dim() == 2 and x2.dtype == torch.bfloat16
            and w.dtype == torch.bfloat16 and w.dim() == 2 and w.is_contiguous() and x2.stride(1) == 1 and x2.shape[1] == w.shape[1]
            and (bias is None or (bias.device == x2.device and bias.dtype == torch.bfloat16 and bias.is_contiguous()
                                  and bias.shape == w.shape[:1])))


def _mid_takes(x2, w, bias, pair, sums=MID_SUMS, rows=MID_ROWS_BLOCK) -> int:
    """``_mid_splits`` for operands that ``mid_gemm`` reads, else 0."""
    splits = _mid_splits(x2.shape[0], w.shape[0], w.shape[1], pair, sums, rows) if _reads(x2, w, bias) else 0
    return 0 if splits and _followed(x2, w, bias) else splits


def _block_takes(x2, w, bias, pair, sums=MID_SUMS) -> int:
    """``_block_splits`` for operands that ``block_gemm`` reads, else 0."""
    if x2.dim() != 2 or not BLOCK_MIN_ROWS <= x2.shape[0] <= BLOCK_MAX_ROWS_LONG or not _reads(x2, w, bias):
        return 0
    splits = _block_splits(x2.shape[0], w.shape[0], w.shape[1], pair, sums)
    return 0 if splits and _followed(x2, w, bias) else splits


def _mid_gemm(x2, w, bias, pair):
    """Projection of up to a few hundred rows (``csrc/kernels/mid_gemm.hip``), or None where another kernel is the better choice."""
    splits = _mid_takes(x2, w, bias, pair)
    if not splits:
        return None
    return _split_product(_kernels().vpsa_mid_gemm, x2, w, bias, pair, splits)


def _block_proj(x2, w, bias, pair):
    """Projection of about a hundred to a few hundred rows (``csrc/kernels/block_gemm.hip``), or None where another kernel is the better
    choice."""
    splits = _block_takes(x2, w, bias, pair)
    if not splits:
        return None
    return _split_product(_kernels().vpsa_block_proj, x2, w, bias, pair, splits)


def _split_product(entry, x2, w, bias, pair, splits):
    m, n, k = x2.shape[0], w.shape[0], w.shape[1]
    out = torch.empty((m, n // 2 if pair else n), dtype=x2.dtype, device=x2.device)
    ws = torch.empty((splits * m * n,), dtype=torch.float32, device=x2.device) if splits > 1 else None
    rc = entry(_p(x2), c_long(x2.stride(0)), _p(w), _p(bias), _p(out), c_long(out.stride(0)), _p(ws), c_int(m),
               c_int(n), c_int(k), c_int(1 if pair else 0), c_int(splits), _stream())
    return out if rc == 0 else None


def linear_add_norm(x, w, residual, weight, eps):
    """``residual += x @ w.T`` and the norm of the new rows, ``rmsnorm(residual) * weight``, when ``mid_gemm`` splits the product: its
    reduction then makes both.  None (and nothing done) otherwise."""
    return _add_norm("vpsa_mid_gemm_norm", _mid_takes(x, w, None, False, MID_SUMS_NORM), x, w, residual, weight, eps)


def block_add_norm(x, w, residual, weight, eps):
    """As ``linear_add_norm``, for the batches from 97 rows on that ``block_gemm`` takes, or ``mid_gemm`` in two blocks of 128 rows."""
    if x.dim() != 2 or not BLOCK_MIN_ROWS <= x.shape[0] <= BLOCK_MAX_ROWS_LONG:
        return None
    y = _add_norm("vpsa_block_proj_norm", _block_takes(x, w, None, False, MID_SUMS_NORM), x, w, residual, weight, eps)
    if y is None and x.shape[0] > MID_ROWS_BLOCK:
        y = _add_norm("vpsa_mid_gemm_norm", _mid_takes(x, w, None, False, MID_SUMS_NORM, MID_ROWS_LONG), x, w, residual, weight, eps)
    return y


def tile_add_norm(x, w, residual, weight, eps):
    """As ``linear_add_norm``, for products of the prefill GEMM with a split tail: the pass that closes it also makes the norm."""
    m, n = x.shape[0], w.shape[0]
    if (not _tile_takes(x, w, False, residual) or n > 8192 or weight.shape != (n,) or weight.device != x.device or weight.dtype != torch.bfloat16
            or not weight.is_contiguous() or weight.data_ptr() % 8 or tile_tail(m, n, w.shape[1]) <= 1 or _followed(weight)):
        return None
    ws = tail_parts(x.device, _tail_slots(m, n, w.shape[1], False))
    tile_gemm(x, w, residual=residual, out=residual, parts=ws)
    y = torch.empty_like(residual)
    rc = _kernels().vpsa_tile_tail_norm(_p(ws), _p(residual), _p(weight), _p(y), c_int(m), c_int(n), c_int(w.shape[1]), c_float(eps), _stream())
    _check(rc, "tile_tail_norm")
    return y


def _add_norm(entry, splits, x, w, residual, weight, eps):
    m, n = x.shape[0], w.shape[0]
    if (splits < 2 or n > 8192 or residual.shape != (m, n) or residual.dtype != torch.bfloat16 or not residual.is_contiguous()
            or residual.device != x.device or weight.device != x.device or weight.dtype != torch.bfloat16 or weight.shape != (n,)
            or not weight.is_contiguous()):
        return None
    y = torch.empty_like(residual)
    ws = torch.empty((splits * m * n,), dtype=torch.float32, device=x.device)
    rc = getattr(_kernels(), entry)(_p(x), c_long(x.stride(0)), _p(w), _p(residual), _p(weight), _p(y), _p(ws), c_int(m),
                                    c_int(n), c_int(w.shape[1]), c_int(splits), c_float(eps), _stream())
    return y if rc == 0 else None


def decode_qkv(x, w, bias, pool, layer, positions, slots, cos_sin, n_q, n_kv):
    """q / k / v projection, rotary embedding and cache write of one token per sequence, when ``mid_gemm`` or ``block_gemm``
    splits the projection: its reduction then rotates and writes the cache.  The query rows [T, n_q * 128], or None (and nothing done)
    otherwise."""
    # block_gemm first, as in the projections by themselves: up to 128 rows it takes what is too large for mid_gemm (10240 x 8192 with the cache, 97
    # rows 41.7 us, with mid_gemm 44.8, 128 rows 44.9 and 50.0; projection and cache's own kernel 44.1 and 46.9)
    splits, entry = _block_takes(x, w, bias, False, BLOCK_SUMS_QKV), "vpsa_block_proj_qkv"
    if splits < 2:
        splits, entry = _mid_takes(x, w, bias, False), "vpsa_mid_gemm_qkv"
    m = x.shape[0]
    if splits < 2 or pool.dtype != torch.bfloat16 or w.shape[0] != (n_q + 2 * n_kv) * HEAD_DIM_HIP:
        return None
    assert positions.dtype == torch.int32 and slots.dtype == torch.int64 and positions.shape[0] >= m and slots.shape[0] >= m
    assert cos_sin.dtype == torch.float32 and cos_sin.shape[1] == HEAD_DIM_HIP
    q = torch.empty((m, n_q * HEAD_DIM_HIP), dtype=x.dtype, device=x.device)
    ws = torch.empty((splits * m * w.shape[0],), dtype=torch.float32, device=x.device)
    base = pool.data_ptr() + layer * pool.stride(1) * 2
    rc = getattr(_kernels(), entry)(_p(x), c_long(x.stride(0)), _p(w), _p(bias), _p(q), _p(ws), c_int(m), c_int(w.shape[1]),
                                    c_int(splits), _p(positions), _p(slots), _p(cos_sin), c_void_p(base), c_long(pool.stride(0)),
                                    c_long(pool.stride(2)), c_int(n_q), c_int(n_kv), _stream())
    return q if rc == 0 else None


def decode_attention_block(x, w, bias, pool, layer, meta, n_q, n_kv, head_dim, scale, cos_sin):
    """Projection, rotary embedding, cache write and attention of a decode-only step where ``decode_qkv`` takes the first three.
    [T, n_q * head_dim], or None (and nothing done) otherwise."""
    if isinstance(pool, LayerGroupedPool):
        pool, layer = pool.for_layer(layer)
    if (meta.num_prefill_seqs > 0 or meta.num_decode != x.shape[0] or meta.slots is None or head_dim != HEAD_DIM_HIP
            or _generic_attention(x, head_dim)):
        return None
    q = decode_qkv(x, w, bias, pool, layer, meta.positions, meta.slots, cos_sin, n_q, n_kv)
    if q is None:
        return None
    out = torch.empty_like(q)
    paged_decode(q, out, pool, layer, meta.dec_block_tables, meta.dec_ctx_lens, n_q, n_kv, head_dim, scale,
                 getattr(meta, "dec_num_splits", 1) or 1, getattr(meta, "dec_ws_o", None), getattr(meta, "dec_ws_ml", None))
    return out


# ``row_gemm``'s products of a few rows (whole in one launch; what closes the one before and opens the next is made beside them) against
# ``mid_gemm``'s, whose reductions are launches of their own, microseconds in a graph over weights that no cache holds (mid / row; q | k | v with
# rotation and cache, output projections with the stream's update and the norm, gated unit):
#   hidden 4096, 14336 wide    1 row 13.9/12.4  11.6/9.2   38.9/39.7  23.9/20.8    8 rows 14.5/12.8  11.9/9.3  38.8/39.3  24.6/21.2    16 rows 15.2/15.4  12.6/10.5  38.9/39.5  25.2/24.4
#   3584, 18944                1     11.0/10.8  10.6/8.3   51.0/57.0  28.1/24.7    8      11.6/11.5  11.1/8.7  52.8/57.4  28.8/26.8    (296 workgroups: a second round)
#   8192, 28672                1     33.2/31.6  29.2/25.8  149/150    79.2/74.3    16     33.8/37.6  29.9/28.5  148/150    79.5/92.7
# A step of 8 layers (hidden 4096): 1 sequence 899 / 880, 2 936 / 877, 4 1098 / 1034, 8 1053 / 1006, 12 1118 / 1095, 14 1069 / 1047, 16 1072 / 1072.
# Other widths have 16 of the hidden rows a workgroup in more than one round, and the last one is as long as the others: a step of 6 layers, before / with
# them: 5120 wide (320 of 512 workgroups) 1 row 714 / 713 us, 8 rows 747 / 770, 14 rows 783 / 852; 6144 (384) 1 row 2.5 % ahead, 8 955 / 953, 9 968 / 974, 14 991 / 1032; 7168
# (448) 8 rows 2.1 % ahead, 9 0.4 %, 11 999 / 1011, 14 1012 / 1048; 8192 (whole rounds) 1 row 3.6 % ahead, 14 1.2; 3072, 3584 and 4096 (one round) 14 rows 2.1 to 3.7 %.
ROW_ROWS = 14
ROW_ROWS_PART = 8   # where a last round is from ROW_PART on, but not nearly, full: up to 8 token rows go through LDS in one group
ROW_PART = 0.75


def row_limit(hidden: int) -> int:
    """Rows up to which a decode step takes ``row_gemm``'s products at a width."""
    tiles = hidden // 16
    fill = tiles / (-(-tiles // TILE_CUS) * TILE_CUS)
    return ROW_ROWS if tiles <= TILE_CUS or fill > 0.95 else ROW_ROWS_PART if fill >= ROW_PART else 0


def row_layer_takes(residual, lw, pool, meta, n_q, n_kv, head_dim, cos_sin) -> bool:
    """Whether a decoder layer of a decode step takes ``row_gemm``'s products: few rows, projections that fill three quarters of the chip's
    workgroups (``row_limit``), a gated unit in one round of them, operands that the kernels read."""
    m, h = residual.shape
    if isinstance(pool, LayerGroupedPool):
        pool = pool.groups[0]
    if (m > min(ROW_ROWS, row_limit(h)) or not residual.is_cuda or head_dim != HEAD_DIM_HIP or meta.slots is None or meta.num_decode != m or meta.num_prefill_seqs > 0
            or lw.w_gate_up is None or lw.w_gate_up_p is not None or lw.w_down_p is not None or pool.dtype != torch.bfloat16
            or _generic_attention(residual, head_dim) or h > 8192):
        return False
    q, i = n_q * head_dim, lw.w_down.shape[1]
    if (h // 16 < MID_MIN_FILL_ROWS or not MID_MIN_FILL_ROWS <= i // 64 <= TILE_CUS or lw.wqkv.shape != (q + 2 * n_kv * head_dim, h)
            or lw.wo.shape != (h, q) or lw.w_gate_up.shape != (2 * i, h) or lw.w_down.shape != (h, i)
            or int(_kernels().vpsa_mid_gemm_splits(c_int(m), c_int(2 * i), c_int(h), c_int(1))) != 1):
        return False
    lib = _kernels()
    if not all(lib.vpsa_row_gemm_takes(c_int(m), c_int(w.shape[0]), c_int(w.shape[1])) for w in (lw.wqkv, lw.wo, lw.w_down)):
        return False
    norms = [t for t in (lw.ln1, lw.ln2) if t.shape == (h,) and t.is_contiguous()]
    if not _reads(residual, lw.wqkv, lw.bqkv) or not _reads(residual, lw.w_gate_up, None) or len(norms) < 2 or not residual.is_contiguous():
        return False
    ws = (lw.wo, lw.w_down)
    return (all(w.dtype == torch.bfloat16 and w.is_contiguous() and w.device == residual.device for w in ws)
            and all(_lies_with(residual, t) for t in (residual, *norms, lw.wqkv, lw.wo, lw.w_gate_up, lw.w_down))
            and (lw.bqkv is None or lw.bqkv.data_ptr() % 8 == 0) and cos_sin.data_ptr() % 16 == 0
            and not _followed(residual, lw.wqkv, lw.bqkv, lw.wo, lw.w_gate_up, lw.w_down, *norms))


def row_add(x, w, residual, norm):
    """``residual += x @ w.T``; with ``norm`` also what the next product starts from: (the new rows times it, sums of 16 of their squares each)."""
    m, n = residual.shape
    assert x.shape == (m, w.shape[1]) and x.stride(1) == 1 and w.shape[0] == n
    normed, squares = None, None
    if norm is not None:
        normed, squares = torch.empty_like(residual), torch.empty((m, n // 16), dtype=torch.float32, device=x.device)
    _check(_kernels().vpsa_row_add(_p(x), c_long(x.stride(0)), _p(w), _p(residual), _p(norm), _p(normed), _p(squares), c_int(m), c_int(n),
                                   c_int(w.shape[1]), _stream()), "row_add")
    return normed, squares


def row_gate_up(rows, eps, w):
    """The gated unit of ``row_add``'s rows, normed."""
    normed, squares = rows
    m, k = normed.shape
    y = torch.empty((m, w.shape[0] // 2), dtype=normed.dtype, device=normed.device)
    _check(_kernels().vpsa_mid_unit_factors(_p(normed), c_long(k), _p(squares), c_float(eps), _p(w), _p(y), c_long(y.stride(0)), c_int(m),
                                            c_int(w.shape[0]), c_int(k), _stream()), "row_gate_up")
    return y


def row_attention_block(rows, eps, w, bias, pool, layer, meta, n_q, n_kv, head_dim, scale, cos_sin):
    """``decode_attention_block`` of ``row_add``'s rows, normed."""
    if isinstance(pool, LayerGroupedPool):
        pool, layer = pool.for_layer(layer)
    normed, squares = rows
    m, k = normed.shape
    assert meta.positions.dtype == torch.int32 and meta.slots.dtype == torch.int64 and min(meta.positions.shape[0], meta.slots.shape[0]) >= m
    assert cos_sin.dtype == torch.float32 and cos_sin.shape[1] == HEAD_DIM_HIP
    q = torch.empty((m, n_q * HEAD_DIM_HIP), dtype=normed.dtype, device=normed.device)
    base = pool.data_ptr() + layer * pool.stride(1) * 2
    _check(_kernels().vpsa_row_qkv(_p(normed), c_long(k), _p(squares), c_float(eps), _p(w), _p(bias), _p(q), c_int(m), c_int(k), _p(meta.positions),
                                   _p(meta.slots), _p(cos_sin), c_void_p(base), c_long(pool.stride(0)), c_long(pool.stride(2)), c_int(n_q),
                                   c_int(n_kv), _stream()), "row_qkv")
    out = torch.empty_like(q)
    paged_decode(q, out, pool, layer, meta.dec_block_tables, meta.dec_ctx_lens, n_q, n_kv, head_dim, scale,
                 getattr(meta, "dec_num_splits", 1) or 1, getattr(meta, "dec_ws_o", None), getattr(meta, "dec_ws_ml", None))
    return out


# The projection's reduction also rotates and writes the cache: a launch less a layer.  A step of 8 layers, apart / together: 32 rows behind
# 1500 tokens 1121 / 1084 us, 64 behind 3000 1270 / 1221, 97 behind 20900 1650 / 1601, 150 behind 3000 1577 / 1534, 256 behind 2000 1818 / 1701; with two
# row tiles 300 behind 1500 2152 / 2122, but 400 2221 / 2274, 512 2488 / 2512: the cache's own kernel writes whole lines of V, the reduction single values.
# Other widths, a step of 4 layers behind 1500 tokens: 28 + 4 heads of 3584 channels with a bias, 16 rows 729 / 714, 80 898 / 876, 129 1003 / 982, 176 1027 / 1020, 240
# 1140 / 1136, 256 1183 / 1125; 64 + 8 of 8192, 16 rows 1556 / 1537, 64 1805 / 1786, 112 1879 / 1855, 128 1935 / 1922, 224 2195 / 2186, 256 2388 / 2407 (runs differ by
# 2 %; projection and cache alone 59.4 / 58.2); 32 + 4 of 8192, 128 rows 1331 / 1294, 256 1543 / 1473; 16 + 2 of 8192, 256 rows 1334 / 1271; 16 + 4 of 4096, 176 rows 763 / 751.
PROMPT_QKV_ROWS = BLOCK_MAX_ROWS


def prompt_attention_block(x, w, bias, pool, layer, meta, n_q, n_kv, head_dim, scale, cos_sin):
    """As ``decode_attention_block`` for a short step with prompt rows, behind decode rows or by themselves."""
    if isinstance(pool, LayerGroupedPool):
        pool, layer = pool.for_layer(layer)
    nd = meta.num_decode
    if (meta.num_prefill_seqs <= 0 or x.dim() != 2 or x.shape[0] > PROMPT_QKV_ROWS or meta.slots is None or head_dim != HEAD_DIM_HIP
            or _generic_attention(x, head_dim)):
        return None
    q = decode_qkv(x, w, bias, pool, layer, meta.positions, meta.slots, cos_sin, n_q, n_kv)
    if q is None:
        return None
    out = (torch.zeros_like if getattr(meta, "pre_padded", False) else torch.empty_like)(q)
    if nd > 0:
        paged_decode(q[:nd], out[:nd], pool, layer, meta.dec_block_tables, meta.dec_ctx_lens, n_q, n_kv, head_dim, scale,
                     getattr(meta, "dec_num_splits", 1) or 1, getattr(meta, "dec_ws_o", None), getattr(meta, "dec_ws_ml", None))
    paged_prefill(q[nd:], out[nd:], pool, layer, meta.pre_block_tables, meta.pre_cu_q, meta.pre_ctx_lens, meta.pre_tile_seq,
                  meta.pre_tile_q0, n_q, n_kv, head_dim, scale, meta.pre_tile_rows, split=getattr(meta, "pre_split", None),
                  split_ws=getattr(meta, "pre_split_ws", None), groups=getattr(meta, "pre_split_groups", None))
    return out


def block_linear(x, ws, biases, gelu=False, residual=None, out=None):
    """act(x @ w.T + bias) (+ residual) for one to three weights of one shape, side by side in the last dimension
    (``csrc/kernels/block_gemm.hip``).  x [B, T, K] with unit stride along K (rows may overlap, as a convolution's unfolded input
    does); ``biases``: one or None for each weight; ``gelu``: its erf form; ``residual`` [B, T, N] or [T, N], added behind the
    activation; ``out`` [B, T, N * len(ws)], may be ``residual``.  None (and nothing done) for operands the kernel does not take."""
    b, t, k = x.shape
    n = ws[0].shape[0]
    res = residual if residual is None or residual.dim() == 3 else residual.unsqueeze(0).expand(b, -1, -1)
    dev = x.device
    for v in (x, res, out, *ws, *biases):
        if v is not None and (v.dtype is not torch.bfloat16 or v.device != dev or v.stride(-1) != 1):
            return None
    if not x.is_cuda or (res is not None and (res.shape != (b, t, n) or len(ws) > 1)):
        return None
    for w in ws:
        if w.shape != (n, k) or w.stride(0) != k:
            return None
    for v in biases:
        if v is not None and v.shape != (n,):
            return None
    if out is None:
        out = torch.empty((b, t, n * len(ws)), dtype=x.dtype, device=dev)
    assert out.shape == (b, t, n * len(ws))
    w, v = [u.data_ptr() for u in ws] + [None, None], [_at(u) for u in biases] + [None, None]
    xs, os_, rs = x.stride(), out.stride(), (0, 0) if res is None else res.stride()
    rc = _kernels().vpsa_block_gemm(x.data_ptr(), xs[1], xs[0], w[0], w[1], w[2], v[0], v[1], v[2], len(ws), out.data_ptr(), os_[1], os_[0],
                                    _at(res), rs[1], rs[0], t, b * t, n, k, 1 if gelu else 0, _raw_stream())
    return out if rc == 0 else None


def pack_weight(w: torch.Tensor) -> torch.Tensor:
    """[N, K] -> the same matrix in matrix-core tile order, [N / 16][K / 32][16][32] flattened
    (N a multiple of 16, K of 32): what ``packed_linear`` streams.  A second copy of the weight."""
    n, k = w.shape
    assert n % 16 == 0 and k % 32 == 0
    return w.view(n // 16, 16, k // 32, 32).permute(0, 2, 1, 3).contiguous().view(-1)


def set_packed_target(workgroups: int) -> int:
    """Workgroups (row blocks x reduction slices) the packed kernel aims for; returns the previous value."""
    return int(_kernels().vpsa_set_packed_target(c_int(workgroups)))


def packed_supported(n: int, k: int, pair: bool = False) -> bool:
    return int(_kernels().vpsa_packed_gemm_splits(c_int(n), c_int(k), c_int(1 if pair else 0))) > 0


def packed_linear(x2, wp, n: int, k: int, bias=None, pair: bool = False):
    """y = x2 @ W.T (+ bias), or silu(x2 @ Wg.T) * (x2 @ Wu.T) for ``pair`` (W = [Wg; Wu]), with W
    given as ``pack_weight(W)``; up to 64 rows.  ``None`` when the kernel does not tile the shape."""
    lib = _kernels()
    m = x2.shape[0]
    splits = int(lib.vpsa_packed_gemm_splits(c_int(n), c_int(k), c_int(1 if pair else 0)))
    if splits <= 0 or m > 64:
        return None
    out = torch.empty((m, n // 2 if pair else n), dtype=x2.dtype, device=x2.device)
    ws = torch.empty((splits * m * n,), dtype=torch.float32, device=x2.device) if splits > 1 else None
    rc = lib.vpsa_packed_gemm(_p(x2), c_long(x2.stride(0)), _p(wp), _p(bias), _p(out), c_long(out.stride(0)),
                              _p(ws), c_int(m), c_int(n), c_int(k), c_int(1 if pair else 0), c_int(splits),
                              _stream())
    return out if rc == 0 else None


def _skinny_ok(x, w, bias):
    return (_skinny_enabled and x.is_cuda and w.device == x.device and x.dtype == torch.bfloat16 and w.dtype == torch.bfloat16
            and w.is_contiguous() and x.dim() == 2 and 0 < x.shape[0] <= SKINNY_MAX_ROWS and x.stride(1) == 1
            and (bias is None or (bias.device == x.device and bias.dtype == torch.bfloat16 and bias.is_contiguous()))
            and not _followed(x, w, bias))


# Dispatch thresholds of shapes that mid_gemm below does not take, measured on MI355X (profiles/gemm_micro_graph.jsonl, HIP-graph replay,
# Llama-3-8B shapes, microseconds: library / register-direct / streaming kernel):
#   o-proj  4096x4096   1-16 rows: 14.9-15.0 /  9.6-11.4 / 11.1-14.4   -> register-direct
#   qkv     6144x4096   1-16 rows: 14.2      / 14.0-19.2 / 12.8-14.0   -> streaming
#   gate_up 28672x4096  1-16 rows: 60.8-61.9 (+ activation) / 55.7-63 / 41.3-45.2; 24-32 rows:
#                                  55 / - / 48.5-49.3; 40 rows: 53.5-55.4 / - / 52.7; 48 rows (where
#                                  the library's pick is a poor one): 63-65 / - / 53.7; 64 rows:
#                                  54.7 / - / 58.5                       -> streaming up to 48 rows
#   lm_head 128256x4096 1-16 rows: 187-189   / 209-288   / 173-184     -> streaming
#   down    4096x14336: the library wins at every batch (24.8 vs 25.6)  -> library
# From ~24 rows on (40 rows: qkv 17 vs 21, o 13 vs 18, down 36 vs 37) the library GEMM is as good or better.
SMALL_BATCH_ROWS = 16
PACKED_MAX_ROWS = 64
PAIR_STREAM_MAX_ROWS = 48
DIRECT_MAX_WEIGHT_ELEMS = 4096 * 4096
STREAM_MAX_K = 8192


# The prefill GEMM (``tile_gemm``: 256 x 256 tiles, one workgroup per CU) is used when its tiles fill
# the chip's 256 CUs in whole rounds: measured on MI355X against the library at 8192 rows 0.95-0.98x
# plain, 1.08x with the SwiGLU epilogue fused (profiles/r3_tile_gemm_micro_v1.jsonl).  Where they do not,
# ``_tile_takes`` looks at what the cut tail saves.
TILE_MIN_ROWS = int(os.environ.get("VPSA_TILE_MIN_ROWS", "1024"))
TILE_MIN_FILL = float(os.environ.get("VPSA_TILE_MIN_FILL", "0.85"))
TILE_CUS = 256
_tile_enabled = os.environ.get("VPSA_TILE_GEMM", "1") != "0"


TILE_GELU_GLU = True  # the gated gelu unit in the prefill GEMM's epilogue (tile_gemm(gelu_mul=True))


def set_tile_gemm(on: bool) -> bool:
    """Switch the hand-written prefill GEMM on or off (A/B timing); returns the old value."""
    global _tile_enabled
    old, _tile_enabled = _tile_enabled, bool(on)
    return old


_shape_log = {} if os.environ.get("VPSA_SHAPE_LOG") else None
if _shape_log is not None:
    import atexit
    import sys
    atexit.register(lambda: print("VPSA_SHAPE_LOG", sorted(_shape_log.items(), key=lambda kv: -kv[1])[:60], file=sys.stderr, flush=True))


def _tile_reads(x, w, *others) -> bool:
    """Whether the prefill GEMM may read these operands, whatever its sizes: a call that something follows from outside is left to the library
    before any address is read (a function transform's tensors have none), and so is what does not lie on the 16 bytes of its
    loads or beyond their 32-bit offsets.  ``others``: a bias [N] or residual [M, N] that the epilogue adds, or None."""
    m, n = x.shape[0], w.shape[0]
    return (x.shape[1] == w.shape[1] and x.stride(1) == 1 and x.stride(0) % 8 == 0
            and w.is_contiguous() and m * x.stride(0) < 1 << 31 and not _followed(x, w, *others)
            and all(t is None or (t.shape == ((n,) if t.dim() == 1 else (m, n)) and t.is_contiguous()) for t in others)
            and all(t is None or _lies_with(x, t) for t in (x, w, *others)))


def _tile_fills(m: int, n: int, k: int, pair: bool) -> bool:
    """Whether whole tiles of these sizes fill their rounds."""
    if _shape_log is not None:
        _shape_log[(m, n, k)] = _shape_log.get((m, n, k), 0) + 1
    if m < TILE_MIN_ROWS or not tile_gemm_supported(n, k, pair):
        return False
    tiles = _tiles(m, n, pair)
    return tiles / (-(-tiles // TILE_CUS) * TILE_CUS) >= TILE_MIN_FILL


def tile_rows(x, w, pair: bool = False) -> int:
    """How many leading rows of ``x`` the prefill GEMM should take for ``x @ w.T``: all of them
    (a ragged last row tile is handled inside the kernel; a separate small GEMM for the remainder
    costs more than the padding), or 0 when the library is the better choice for this shape."""
    if not (_tile_enabled and x.is_cuda and x.dim() == w.dim() == 2) or not _tile_fills(x.shape[0], *w.shape, pair):
        return 0
    return x.shape[0] if _tile_reads(x, w) else 0


# With the last round's tiles cut (``tile_tail``) and the activation in the epilogue the kernel is ahead of the library at other sizes as
# well, microseconds, library with its activation or norm pass / here (weights that no cache holds):
#   28672 x 4096 pair     257 rows 80/74     512 rows 109/99    700 rows 169/149   1200 rows 282/233    2100 rows 437/390    5300 rows 1044/921
#   57344 x 8192 pair     300      318/304   512      422/369   1000     813/699   1500      1112/1017
#   37888 x 3584 pair     300      121/105   512      150/131   1000     324/232   1500      384/335
#   16384 x 2048 pair     300      36/38     512      42/47     700      54/48     1500      107/96     (300, 512: half a round, short reductions)
#   4096 x 14336, norm    600      124/81    1000     144/107   1500     181/163   2100      249/251    4200      790/401     5300     785/482
#   8192 x 28672, norm    700      331/315   1000     392/351   1500     561/573   2100      1440/751   4200      2066/1411
#   3584 x 18944, norm    700      173/95    1500     281/181   2100     353/249   5300      1089/587
#   2048 x 8192, norm     700      50/47     1500     70/68     3000     101/102
#   10240 x 8192          512      96/88     700      110/106   1000     140/161   2100      304/291
#   6144 x 4096           512      39/48     1000     56/63     3000     139/132   3500      145/148    6000      244/236
#   4096 x 4096, norm     512      35/44     1000     49/55     4200     155/151   5300      173/181    6000      190/196
TILE_TAIL_ROWS = TILE_MIN_ROWS if "VPSA_TILE_MIN_ROWS" in os.environ else 257
TILE_PAIR_FILL = 0.7         # of the rounds, where the kernel also saves the activation's pass
TILE_LONG_CHUNKS = 128       # reductions from which on a product with a cut tail is ahead ...
TILE_TAIL_SPLITS = 4         # ... and elsewhere the ranges that a tail behind whole rounds has


def _tile_takes(x, w, pair: bool = False, *others) -> bool:
    """Whether the prefill GEMM should take all rows of ``x @ w.T``: by size as ``tile_rows`` does, or by the rule above for plain and gated
    products, and in both cases operands that it reads.  ``others``: a bias or residual that the epilogue adds."""
    if not (_tile_enabled and x.is_cuda and x.dim() == w.dim() == 2):
        return False
    m, (n, k) = x.shape[0], w.shape
    return (_tile_fills(m, n, k, pair) or _tile_tail_pays(m, n, k, pair)) and _tile_reads(x, w, *others)


def _tile_tail_pays(m: int, n: int, k: int, pair: bool) -> bool:
    """The rule above, for sizes."""
    if m < TILE_TAIL_ROWS or not tile_gemm_supported(n, k, pair):
        return False
    tiles, splits = -(-m // 256) * (-(-n // 256)), tile_tail(m, n, k, pair)
    if pair:
        return splits > 1 and tiles >= TILE_CUS or tiles >= TILE_PAIR_FILL * TILE_CUS * -(-tiles // TILE_CUS)
    return splits > 1 and (k >= 64 * TILE_LONG_CHUNKS or (tiles >= TILE_CUS and splits >= TILE_TAIL_SPLITS))


def linear(x, w, bias=None, packed=None):
    """y = x @ w.T (+ bias).  Prefill-sized batches run the hand-written 256 x 256 MFMA kernel
    (``csrc/kernels/tile_gemm.hip``) when its tiles fill the chip; batches of up to a hundred rows or so ``mid_gemm.hip``
    and of up to a few hundred ``block_gemm.hip`` where their workgroups do (``_mid_splits``, ``_block_splits``), of up to 16 rows otherwise
    the weight-streaming MFMA kernels of ``csrc/kernels/gemm.hip`` (which one depends on the
    weight's shape); everything else goes to the library GEMM (hipBLASLt).  ``packed``:
    ``pack_weight(w)`` when the caller keeps one (decode-only steps): up to 64 rows then stream
    that copy."""
    if packed is not None and x.dim() == 2 and x.shape[0] <= PACKED_MAX_ROWS and _skinny_ok(x, w, bias):
        y = packed_linear(x, packed, w.shape[0], w.shape[1], bias, False)
        if y is not None:
            return y
    y = _block_proj(x, w, bias, False)
    if y is None:
        y = _mid_gemm(x, w, bias, False)
    if y is not None:
        return y
    if x.dim() == 2 and x.shape[0] <= SMALL_BATCH_ROWS and _skinny_ok(x, w, bias):
        y = None
        if w.numel() <= DIRECT_MAX_WEIGHT_ELEMS:
            y = _skinny(x, w, bias, False)
        elif w.shape[1] <= STREAM_MAX_K:
            y = _stream_gemm(x, w, bias, False)
        if y is not None:
            return y
    if _tile_takes(x, w, False, bias):
        # a bias is a "residual" with row stride 0
        return tile_gemm(x, w, residual=None if bias is None else bias.view(1, -1).expand(x.shape[0], -1))
    return torch.nn.functional.linear(x, w, bias)


def linear_add(x, w, residual, packed=None):
    """The residual-stream update of an output projection: ``residual += x @ w.T`` inside the GEMM's
    epilogue when the prefill kernel takes the shape (returns None: nothing is left to add), else
    returns ``x @ w.T`` for the caller's fused add + norm."""
    if not _tile_takes(x, w, False, residual):
        return linear(x, w, None, packed)
    tile_gemm(x, w, residual=residual, out=residual)
    return None


# The library's pick for the fused q/k/v width of Llama-3-8B (6144 columns) is 12-14 % slower per
# column than its pick for 4096 and 2048 columns at 8192 rows, 7 % at 4096 rows, and faster below
# (profiles/r2_gemm_split_probe.jsonl); other projections gain nothing from a split.
SPLIT_QKV_MIN_ROWS = 4096


def qkv_linear(x, w, bias, q_cols: int):
    """The fused q/k/v projection: ``linear``, except that prefill-sized batches which the
    hand-written kernel does not take and that have no bias go to the library as two GEMMs,
    [q | k v], each writing its column range of ONE output buffer (same bits as the single call)."""
    if (bias is None and x.is_cuda and x.dim() == 2 and x.shape[0] >= SPLIT_QKV_MIN_ROWS
            and x.dtype == torch.bfloat16 and 0 < q_cols < w.shape[0] and not _tile_takes(x, w) and not _followed(x, w)):
        out = torch.empty((x.shape[0], w.shape[0]), dtype=x.dtype, device=x.device)
        torch.matmul(x, w[:q_cols].t(), out=out[:, :q_cols])
        torch.matmul(x, w[q_cols:].t(), out=out[:, q_cols:])
        return out
    return linear(x, w, bias)


def gate_up_silu(x, w_gate_up, packed=None):
    """silu(x @ Wg.T) * (x @ Wu.T) for ``w_gate_up = [Wg; Wu]``: fused in one kernel for
    batches of up to a hundred rows or so (``mid_gemm`` and the weight-streaming kernels) and for prefill batches (SwiGLU epilogue of the 256 x 256
    MFMA kernel); library GEMM + activation kernel for what neither takes.  ``packed`` as in ``linear``."""
    if packed is not None and x.dim() == 2 and x.shape[0] <= PACKED_MAX_ROWS and _skinny_ok(x, w_gate_up, None):
        y = packed_linear(x, packed, w_gate_up.shape[0], w_gate_up.shape[1], None, True)
        if y is not None:
            return y
    y = _block_proj(x, w_gate_up, None, True)
    if y is None:
        y = _mid_gemm(x, w_gate_up, None, True)
    if y is not None:
        return y
    if x.dim() == 2 and x.shape[0] <= PAIR_STREAM_MAX_ROWS and _skinny_ok(x, w_gate_up, None):
        y = _stream_gemm(x, w_gate_up, None, True)
        if y is None and x.shape[0] <= 8:
            y = _skinny(x, w_gate_up, None, True)
        if y is not None:
            return y
    if _tile_takes(x, w_gate_up, True):
        return tile_gemm(x, w_gate_up, silu_mul=True)
    return silu_and_mul(torch.nn.functional.linear(x, w_gate_up))


def hbm_read_probe(buf, blocks=2048):
    """Launch the read-bandwidth probe over ``buf`` (timing is the caller's)."""
    sink = torch.zeros(1, dtype=torch.int32, device=buf.device)
    rc = _kernels().vpsa_hbm_read_probe(_p(buf), c_long(buf.numel() * buf.element_size()), _p(sink),
                                        c_int(blocks), _stream())
    _check(rc, "hbm_read_probe")


# --------------------------------------------------------------------------- MLP / sampling
def silu_and_mul(x, out=None):
    if not x.is_cuda or (out is None and _followed(x)):
        y = reference.silu_and_mul(x)
        if out is not None:
            out.copy_(y)
            return out
        return y
    _bf16_cuda(x)
    inter = x.shape[-1] // 2
    x2 = x.view(-1, 2 * inter)
    assert x2.is_contiguous()
    if out is None:
        out = torch.empty((x2.shape[0], inter), dtype=x.dtype, device=x.device)
    rc = _kernels().vpsa_silu_mul(_p(x2), _p(out), c_long(x2.shape[0]), c_int(inter), _stream())
    _check(rc, "silu_and_mul")
    return out.view(*x.shape[:-1], inter)


def argmax(logits, out=None):
    if not logits.is_cuda:
        return reference.argmax(logits)
    if logits.dtype != torch.bfloat16 or logits.stride(-1) != 1 or logits.stride(0) % 8 != 0:
        return torch.argmax(logits, dim=-1)
    if out is None:
        out = torch.empty((logits.shape[0],), dtype=torch.int64, device=logits.device)
    rc = _kernels().vpsa_argmax_bf16(_p(logits), _p(out), c_int(logits.shape[0]),
                                     c_int(logits.shape[1]), c_long(logits.stride(0)), _stream())
    _check(rc, "argmax")
    return out


def sample_supported(logits) -> bool:
    return (logits.is_cuda and logits.dtype == torch.bfloat16 and logits.dim() == 2
            and logits.stride(1) == 1 and logits.stride(0) % 8 == 0 and logits.data_ptr() % 16 == 0)


def sample(logits, params, uniform, rows=None, want_stats=False):
    """Draw one token per sample from bf16 ``logits`` [*, vocab] in one launch.
    ``params`` float32 [n, 3] = (temperature, top_p, top_k; top_k <= 0 and top_p >= 1 mean off),
    ``uniform`` float32 [n] in [0, 1), ``rows`` int32 [n] (logits row of each sample; default
    sample i reads row i).  -> int64 token ids [n] (and, for tests, [n, 3] = threshold key,
    kept mass relative to the largest probability, kept count)."""
    if not sample_supported(logits):
        raise TypeError("sample: bf16 device logits with 16-byte aligned rows")
    n = params.shape[0]
    out = torch.empty((n,), dtype=torch.int64, device=logits.device)
    stats = torch.empty((n, 3), dtype=torch.float32, device=logits.device) if want_stats else None
    assert params.dtype == torch.float32 and params.is_contiguous() and uniform.dtype == torch.float32
    assert rows is None or (rows.dtype == torch.int32 and rows.numel() == n)
    rc = _kernels().vpsa_sample(_p(logits), c_long(logits.stride(0)), c_int(logits.shape[1]), _p(rows),
                                _p(params), _p(uniform), _p(out), _p(stats), c_int(n), _stream())
    _check(rc, "sample")
    return (out, stats) if want_stats else out


# --------------------------------------------------------------------------- KV page movement
def kv_gather_pages(pool, page_ids, staging):
    """Copy whole pages (all layers) ``pool[page_ids]`` into contiguous ``staging``."""
    if not pool.is_cuda:
        staging.view(-1)[: page_ids.numel() * pool[0].numel()].view(page_ids.numel(), -1).copy_(
            pool[page_ids.long()].reshape(page_ids.numel(), -1))
        return
    assert page_ids.dtype == torch.int64 and page_ids.is_cuda
    page_bytes = pool.stride(0) * pool.element_size()
    assert staging.numel() * staging.element_size() >= page_ids.numel() * page_bytes
    rc = _kernels().vpsa_kv_gather_pages(_p(pool), _p(page_ids), _p(staging),
                                         c_int(page_ids.numel()), c_long(page_bytes), _stream())
    _check(rc, "kv_gather_pages")


def kv_scatter_pages(staging, page_ids, pool):
    if not pool.is_cuda:
        pool[page_ids.long()] = staging.view(-1)[: page_ids.numel() * pool[0].numel()].view(
            page_ids.numel(), *pool.shape[1:]).to(pool.dtype)
        return
    assert page_ids.dtype == torch.int64 and page_ids.is_cuda
    page_bytes = pool.stride(0) * pool.element_size()
    rc = _kernels().vpsa_kv_scatter_pages(_p(staging), _p(page_ids), _p(pool),
                                          c_int(page_ids.numel()), c_long(page_bytes), _stream())
    _check(rc, "kv_scatter_pages")


def cachegen_encode(staging, levels, unit_elems, n_layers, scales=None):
    """bf16 staging -> (int8 symbols, fp32 group scales, in ``scales`` where given).  ``levels``: int32 tensor [n_layers]."""
    if not staging.is_cuda:
        sym, sc = reference.cachegen_encode(staging, levels.tolist(), unit_elems, n_layers)
        return sym, sc if scales is None else scales.copy_(sc)
    n = staging.numel()
    sym = torch.empty((n,), dtype=torch.int8, device=staging.device)
    if scales is None:
        scales = torch.empty((n // 64,), dtype=torch.float32, device=staging.device)
    assert scales.dtype == torch.float32 and scales.is_contiguous() and scales.numel() == n // 64
    assert levels.dtype == torch.int32 and levels.is_cuda
    rc = _kernels().vpsa_cachegen_encode(_p(staging), _p(sym), _p(scales), _p(levels), c_long(n),
                                         c_long(unit_elems), c_int(n_layers), _stream())
    _check(rc, "cachegen_encode")
    return sym, scales


def cachegen_decode(symbols, scales, unit_elems, out=None):
    if not symbols.is_cuda:
        y = reference.cachegen_decode(symbols, scales, unit_elems)
        if out is not None:
            out.view(-1).copy_(y)
            return out
        return y
    n = symbols.numel()
    if out is None:
        out = torch.empty((n,), dtype=torch.bfloat16, device=symbols.device)
    rc = _kernels().vpsa_cachegen_decode(_p(symbols), _p(scales), _p(out), c_long(n),
                                         c_long(unit_elems), _stream())
    _check(rc, "cachegen_decode")
    return out


# --------------------------------------------------------------------------- rANS entropy stage
RANS_SPC = 512  # streams per context: 256 symbols per stream for a Llama-3-8B layer (K + V)


def rans_encode(sym, n_ctx, spc=RANS_SPC):
    """Entropy-code int8/uint8 symbols (``n_ctx`` equal contexts) with the interleaved rANS
    coder.  -> (freq int16 [n_ctx * 256], states int32 [n_ctx * spc], sizes int16 [n_ctx * spc],
    coded uint8 [sum of sizes]); the 16/32-bit tensors hold unsigned values bit for bit.
    Synchronises once (the coded length sizes the output)."""
    if not sym.is_cuda:
        import numpy as np

        f, st, sz, co = reference.rans_encode(sym.contiguous().view(torch.uint8).numpy(), n_ctx, spc)
        return (torch.from_numpy(f.view(np.int16).reshape(-1).copy()), torch.from_numpy(st.view(np.int32).copy()),
                torch.from_numpy(sz.view(np.int16).copy()), torch.from_numpy(co.copy()))
    sym = sym.contiguous().view(torch.uint8).view(-1)
    if sym.data_ptr() % 4:  # (a slice at an odd offset: the histogram reads words)
        sym = sym.clone()
    n, dev = sym.numel(), sym.device
    n_streams = n_ctx * spc
    freq = torch.empty(n_ctx * 256, dtype=torch.int16, device=dev)
    states = torch.empty(n_streams, dtype=torch.int32, device=dev)
    sizes = torch.empty(n_streams, dtype=torch.int16, device=dev)
    coded = torch.empty(2 * n, dtype=torch.uint8, device=dev)
    total, bad = rans_encode_into(sym, n_ctx, freq, states, sizes, coded, spc).tolist()  # one synchronisation
    if bad:
        raise RuntimeError("rans_encode: frequency table could not be normalised")
    return freq, states, sizes, coded[:total].clone()


def rans_encode_into(sym, n_ctx, freq, states, sizes, coded, spc=RANS_SPC, meta=None):
    """``rans_encode`` on the device into the caller's tensors (``coded`` with room for two bytes a symbol), without a
    synchronisation -> int64 [2] on the device, or ``meta`` (on the device or in pinned host memory): coded bytes, and contexts
    whose table could not be normalised (nothing of the result is valid unless 0)."""
    n, dev, lib = sym.numel(), sym.device, _kernels()
    if n % n_ctx or (n // n_ctx) % spc:
        raise ValueError("rans_encode: symbols do not divide into contexts / streams")
    n_streams = n_ctx * spc
    assert sym.is_cuda and sym.is_contiguous() and sym.element_size() == 1 and sym.data_ptr() % 4 == 0
    assert all(t.is_contiguous() and t.numel() * t.element_size() >= b for t, b in (
        (freq, 512 * n_ctx), (states, 4 * n_streams), (sizes, 2 * n_streams), (coded, 2 * n)))
    ws = torch.empty(max(1, int(lib.vpsa_rans_workspace(c_long(n), c_int(n_ctx), c_int(spc)))), dtype=torch.uint8, device=dev)
    if meta is None:
        meta = torch.empty(2, dtype=torch.int64, device=dev)
    assert meta.dtype == torch.int64 and meta.is_contiguous() and meta.numel() == 2 and (meta.device == dev or meta.is_pinned())
    _check(lib.vpsa_rans_encode(_p(sym), c_long(n), c_int(n_ctx), c_int(spc), _p(ws), _p(freq), _p(states), _p(sizes), _p(coded),
                                _p(meta), _stream()), "rans_encode")
    return meta


def rans_decode(freq, states, sizes, coded, n, n_ctx, spc=RANS_SPC):
    """Inverse of ``rans_encode`` -> int8 symbols [n] on the device of ``coded``."""
    if not coded.is_cuda:
        import numpy as np

        out = reference.rans_decode(freq.numpy().view(np.uint16), states.numpy().view(np.uint32),
                                    sizes.numpy().view(np.uint16), coded.numpy(), n, n_ctx, spc)
        return torch.from_numpy(out.view(np.int8).copy())
    dev = coded.device
    lib = _kernels()
    freq, states, sizes = freq.contiguous(), states.contiguous(), sizes.to(torch.int16).contiguous()
    assert coded.is_contiguous() and freq.numel() >= n_ctx * 256 and min(states.numel(), sizes.numel()) >= n_ctx * spc
    assert freq.element_size() == 2 and states.element_size() == 4 and all(t.device == dev for t in (freq, states, sizes))
    size = int(lib.vpsa_rans_decode_workspace(c_long(n), c_int(n_ctx), c_int(spc)))
    ws = torch.empty(size, dtype=torch.uint8, device=dev) if size else None
    sym = torch.empty(n, dtype=torch.int8, device=dev)
    _check(lib.vpsa_rans_decode(_p(coded), c_long(coded.numel()), _p(states), _p(freq), _p(sizes), _p(ws), _p(sym), c_long(n), c_int(n_ctx),
                                c_int(spc), _stream()), "rans_decode")
    return sym


def fetch_bytes(src, pinned, dst: int, size: int) -> None:
    """The first ``size`` bytes of ``src`` (uint8, on the device) to host memory at ``dst``, through ``pinned`` (as large, pinned): the
    buffer is emptied behind the copy that fills it.  Over on return; other threads run meanwhile."""
    assert src.is_cuda and src.is_contiguous() and min(src.numel(), pinned.numel()) >= size and not pinned.is_cuda
    _check(_kernels().vpsa_fetch(_p(src), _p(pinned), c_void_p(dst), c_long(size), _stream()), "fetch_bytes")


def page_decode(src: int, pinned, size: int, n: int, n_ctx: int, unit_elems: int, device, spc=RANS_SPC):
    """A page's quantised and coded parts (``size`` host bytes at ``src``: scales fp32 [n / 64] | freq u16 [n_ctx * 256] | states u32 and
    sizes u16 [n_ctx * spc] | coded bytes) -> bf16 [n] on ``device``, by way of ``pinned``, which the device reads until what has been
    queued so far is over.  The bytes come into a device buffer that stays with ``pinned`` (its ``body``), from the second page on, on a stream of
    the kernel library's, beside the kernels of the page before: no call may use ``pinned`` again, nor let go of it, before this one is over."""
    lib = _kernels()
    ws = int(lib.vpsa_page_workspace(c_long(n), c_int(n_ctx), c_int(spc)))
    if ws <= 0 or unit_elems % 8192:
        raise ValueError("page_decode: symbols do not divide into contexts / streams")
    assert pinned.numel() >= size and not pinned.is_cuda
    out = torch.empty(n, dtype=torch.bfloat16, device=device)
    work = torch.empty(ws, dtype=torch.uint8, device=device)
    body = getattr(pinned, "body", None)
    fresh = body is None or body.numel() < size or body.device != out.device
    if fresh:
        body = torch.empty(max(size, pinned.numel()), dtype=torch.uint8, device=device)
    _check(lib.vpsa_page_decode(src, pinned.data_ptr(), body.data_ptr(), size, n, n_ctx, spc, unit_elems, work.data_ptr(), out.data_ptr(),
                                int(fresh), _raw_stream()), "page_decode")
    pinned.body = body
    return out


# --------------------------------------------------------------------------- MoE routing
# A router's product of ``csrc/kernels/moe.hip`` beside the library's, microseconds in a graph (library / kernel), which reads 16 rows of
# weights and activations an instruction and has a workgroup for 16 tokens: short rows and few experts are its side, and one round.
#   8 experts of 4096    8 tokens 7.9/6.2    300 tokens 8.1/7.7    4096 tokens 12.0/8.6    6000 tokens 11.6/14.6
#   8 of 6144            8        6.9/8.4    300        7.1/10.6
#   16 of 2048           8        5.3/4.7    300        5.7/5.6    4096         5.9/6.1
#   16 of 4096           8        7.8/7.5    300        8.1/9.0
#   32 of 1024           8        4.7/4.4    300        5.5/5.0    6000         5.7/7.8
#   32 of 4096           8        7.4/11.0   300        7.5/12.6
#   64 of 512            8        4.0/4.0    300        4.5/3.9
#   64 of 2048           8        5.6/10.4   300        5.6/11.3
MOE_ROUTER_WEIGHTS = 32768  # elements, experts rounded up to 8, 16, 32 or 64
MOE_ROUTER_TOKENS = 4096


def moe_router_takes(tokens: int, experts: int, hidden: int) -> bool:
    """Does a router's product run in the framework's kernel?"""
    return (0 < experts <= 64 and hidden % 128 == 0 and tokens <= MOE_ROUTER_TOKENS
            and hidden * (1 << (max(experts, 8) - 1).bit_length()) <= MOE_ROUTER_WEIGHTS)


def moe_router(x, w):
    """A mixture's router product ``x @ w.T`` (``csrc/kernels/moe.hip`` where ``moe_router_takes`` it, else the library)."""
    if (x.is_cuda and x.dim() == 2 and w.device == x.device and x.dtype == torch.bfloat16 and w.dtype == torch.bfloat16 and w.is_contiguous()
            and w.dim() == 2 and x.shape[1] == w.shape[1] and moe_router_takes(x.shape[0], w.shape[0], w.shape[1]) and x.stride(1) == 1
            and x.stride(0) % 8 == 0 and (x.data_ptr() | w.data_ptr()) % 16 == 0 and not _followed(x, w)):
        out = torch.empty((x.shape[0], w.shape[0]), dtype=x.dtype, device=x.device)
        _check(_kernels().vpsa_moe_router(_p(x), c_long(x.stride(0)), _p(w), _p(out), c_int(x.shape[0]), c_int(w.shape[0]),
                                          c_int(x.shape[1]), _stream()), "moe_router")
        return out
    return torch.nn.functional.linear(x, w)


def moe_topk_softmax(logits, topk, renorm=True):
    if not logits.is_cuda:
        return reference.moe_topk_softmax(logits, topk, renorm)
    _bf16_cuda(logits)
    t, e = logits.shape
    w = torch.empty((t, topk), dtype=torch.float32, device=logits.device)
    ids = torch.empty((t, topk), dtype=torch.int32, device=logits.device)
    rc = _kernels().vpsa_moe_topk_softmax(_p(logits.contiguous()), _p(w), _p(ids), c_int(t),
                                          c_int(e), c_int(topk), c_int(1 if renorm else 0),
                                          _stream())
    _check(rc, "moe_topk_softmax")
    return w, ids


def moe_localize(ids, weights, first, count, bucket):
    """Routing of a rank that holds experts ``first .. first + count`` only: ids become local, and a
    pair routed elsewhere gets weight 0 and the id ``count`` (``bucket``: a sorting bucket of its
    own that ``moe_experts_grouped`` / ``moe_experts_prefill`` skip with ``foreign=True``) or 0."""
    local = ids - first
    here = (local >= 0) & (local < count)
    elsewhere = count if bucket else 0
    return (torch.where(here, local, elsewhere).to(torch.int32),
            torch.where(here, weights, 0.0).to(weights.dtype))


def moe_align(ids, n_experts, weights=None):
    """ids [T, K] int32 -> (offsets [E+1], pos [T*K], sorted_tok [T*K]); with ``weights`` (fp32 [T, K]) a fourth:
    the pairs' weights in sorted order."""
    t, k = ids.shape
    if not ids.is_cuda:
        flat = ids.reshape(-1).long()
        order = torch.sort(flat, stable=True).indices
        pos = torch.empty_like(order)
        pos[order] = torch.arange(order.numel())
        counts = torch.bincount(flat, minlength=n_experts)
        offsets = torch.zeros(n_experts + 1, dtype=torch.int32)
        offsets[1:] = counts.cumsum(0)
        out = (offsets, pos.int(), (order // k).int())
        return out if weights is None else (*out, weights.reshape(-1)[order])
    offsets = torch.empty((n_experts + 1,), dtype=torch.int32, device=ids.device)
    pos = torch.empty((t * k,), dtype=torch.int32, device=ids.device)
    sorted_tok = torch.empty((t * k,), dtype=torch.int32, device=ids.device)
    sorted_w = None
    if weights is not None:
        assert weights.dtype == torch.float32 and weights.is_contiguous() and weights.numel() == t * k
        sorted_w = torch.empty((t * k,), dtype=torch.float32, device=ids.device)
    rc = _kernels().vpsa_moe_align(_p(ids.contiguous()), _p(offsets), _p(pos), _p(sorted_tok), _p(weights), _p(sorted_w),
                                   c_int(t * k), c_int(n_experts), c_int(k), _stream())
    _check(rc, "moe_align")
    return (offsets, pos, sorted_tok) if weights is None else (offsets, pos, sorted_tok, sorted_w)


def moe_permute(x, sorted_tok):
    if not x.is_cuda:
        return x[sorted_tok.long()]
    _bf16_cuda(x)
    xs = torch.empty((sorted_tok.numel(), x.shape[1]), dtype=x.dtype, device=x.device)
    rc = _kernels().vpsa_moe_permute(_p(x.contiguous()), _p(sorted_tok), _p(xs),
                                     c_int(sorted_tok.numel()), c_int(x.shape[1]), _stream())
    _check(rc, "moe_permute")
    return xs


def moe_combine(y, weights, pos, tokens):
    k = weights.shape[1]
    if not y.is_cuda:
        g = y[pos.long()].view(tokens, k, -1).float()
        return (g * weights[:, :, None]).sum(1).to(y.dtype)
    _bf16_cuda(y)
    out = torch.empty((tokens, y.shape[1]), dtype=y.dtype, device=y.device)
    rc = _kernels().vpsa_moe_combine(_p(y.contiguous()), _p(weights), _p(pos), _p(out),
                                     c_int(tokens), c_int(y.shape[1]), c_int(k), _stream())
    _check(rc, "moe_combine")
    return out


# Batches whose experts see few rows each take the kernels that stream every routed expert's weights once (``csrc/kernels/mid_gemm.hip``)
# instead of the 256-row tiles: either few tokens, or few rows an expert on average (a pass takes 64).  One mixture, microseconds in a
# graph, tiles / streaming: 8 experts of 28672 x 4096, two a token: 16 tokens 660/435, 48 660/425, 128 674/491, 192 682/619, 224 683/696, 256
# rows of a prompt 730/910; 16 of 2048 x 2048, four a token: 48 66.5/40.6, 192 69.9/46.7, 224 72.0/67.5; 32, four a token: 384 131/112; 64,
# eight a token: 384 251/170; 128: 768 540/323; 256 of 4096 x 2048: 768 2348/1082.  Where one expert sees every token as well (a pass of
# its own for each 64): 8 experts 192 tokens 705/714, 16 90/96, 32 384 185/180, 64 384 317/206, 128 768 618/401.
# VPSA_MOE_MFMA_MAX_TOKENS sets the bound on the tokens and leaves the rows out of it (0: never).
MOE_MFMA_MAX_TOKENS = int(os.environ.get("VPSA_MOE_MFMA_MAX_TOKENS", "48"))
MOE_STREAM_ROWS = 0 if "VPSA_MOE_MFMA_MAX_TOKENS" in os.environ else 48


def moe_streams_experts(tokens: int, topk: int, experts: int) -> bool:
    return tokens <= MOE_MFMA_MAX_TOKENS or (MOE_MFMA_MAX_TOKENS > 0 and tokens * topk <= MOE_STREAM_ROWS * experts)


def moe_mfma_supported(hidden: int, inter: int) -> bool:
    return hidden % 128 == 0 and inter % 512 == 0


def _rows16(x):
    """``x`` contiguous and on a 16-byte boundary (what loads straight into LDS take)."""
    x = x.contiguous()
    return x if x.data_ptr() % 16 == 0 else x.clone()


def moe_experts_grouped(x, w13, w2, ids, weights, foreign=False, combine=True):
    """Expert MLP for a decode-sized batch: out[t] = sum_k weights[t,k] * MLP_{ids[t,k]}(x[t]).
    ``foreign``: ids may equal the expert count (a pair of an expert held by another rank, weight
    0): those pairs sort behind the last expert and no kernel touches them.

    Same contract as ``moe_experts_small_batch``; here the (token, k) pairs are sorted by expert
    first, and each expert's weights are streamed once against all of its tokens on the matrix
    cores.  Three launches after the sort (gate_up+SiLU, down, weighted combine), no host
    synchronisation: HIP-graph capturable."""
    t, k = ids.shape
    if not x.is_cuda:
        return reference.moe_experts(x, w13, w2, ids, weights)
    _bf16_cuda(x, w13, w2)
    n_experts, hidden, inter = w13.shape[0], x.shape[1], w2.shape[2]
    assert w13.shape[1] == 2 * inter and w13.shape[2] == hidden and w2.shape[1] == hidden
    assert w13.is_contiguous() and w2.is_contiguous() and ids.dtype == torch.int32
    assert moe_mfma_supported(hidden, inter), (hidden, inter)
    if t > 1 and t * hidden >= 1 << 31:  # the kernels reach a batch's rows with offsets of 32 bits
        cut = [moe_experts_grouped(x[i], w13, w2, ids[i], None if weights is None else weights[i], foreign, combine)
               for i in (slice(0, t // 2), slice(t // 2, t))]
        if combine:
            return torch.cat(cut)
        return torch.cat([cut[0][0], cut[1][0]]), torch.cat([cut[0][1], cut[1][1] + t // 2 * k])
    x, w13, w2 = _rows16(x), _rows16(w13), _rows16(w2)
    offsets, pos, sorted_tok = moe_align(ids, n_experts + (1 if foreign else 0))
    act = torch.empty((t * k, inter), dtype=x.dtype, device=x.device)
    y = torch.empty((t * k, hidden), dtype=x.dtype, device=x.device)
    rc = _kernels().vpsa_moe_mfma(_p(x), _p(w13), _p(w2), _p(offsets), _p(sorted_tok),
                                  _p(act), _p(y), c_int(t), c_int(k), c_int(n_experts),
                                  c_int(hidden), c_int(inter), _stream())
    _check(rc, "moe_mfma")
    if not combine:  # the caller sums the pairs itself (y in sorted order, pos: the sorted row of pair t * K + k)
        return y, pos
    return moe_combine(y, weights, pos, t)


def grouped_gemm(a, w, offsets, rows=None, arow_idx=None, silu_mul=False, out=None):
    """out[r, :] = a[arow_idx[r] if given else r, :] @ w[g]^T for offsets[g] <= r < offsets[g+1].

    a [*, K] bf16; w [G, N, K] bf16 contiguous; offsets [G + 1] int32 ON THE DEVICE (the host never
    reads them: one launch for all groups, no synchronisation, HIP-graph capturable); rows = upper
    bound on offsets[G] (default: a.shape[0], or len(arow_idx)).  silu_mul: w[g] is [gate rows | up
    rows] and the result is silu(gate) * up, [rows, N / 2].  Rows at or past offsets[G] are left
    unwritten.  CPU tensors take the PyTorch definition of the same product."""
    g, n, k = w.shape
    if rows is None:
        rows = a.shape[0] if arow_idx is None else arow_idx.numel()
    n_out = n // 2 if silu_mul else n
    if not a.is_cuda:
        off = offsets.tolist()
        res = torch.zeros((rows, n_out), dtype=a.dtype) if out is None else out
        src = a if arow_idx is None else a[arow_idx.long()]
        for i in range(g):
            lo, hi = off[i], off[i + 1]
            if hi > lo:
                y = src[lo:hi].float() @ w[i].float().t()
                if silu_mul:
                    y = torch.nn.functional.silu(y[:, :n_out]) * y[:, n_out:]
                res[lo:hi] = y.to(a.dtype)
        return res
    _bf16_cuda(a, w)
    assert w.is_contiguous() and a.stride(-1) == 1 and a.shape[1] == k and offsets.dtype == torch.int32
    assert offsets.numel() == g + 1 and offsets.is_cuda
    if arow_idx is not None:
        assert arow_idx.dtype == torch.int32 and arow_idx.is_cuda and arow_idx.numel() >= rows
    if out is None:
        out = torch.empty((rows, n_out), dtype=a.dtype, device=a.device)
    assert out.stride(-1) == 1 and out.shape[0] >= rows and out.shape[1] == n_out
    rc = _kernels().vpsa_grouped_gemm(_p(a), c_long(a.stride(0)), _p(arow_idx),
                                      _p(w), _p(offsets), c_int(g), _p(out), c_long(out.stride(0)), c_int(rows),
                                      c_int(n), c_int(k), c_int(1 if silu_mul else 0), _stream())
    _check(rc, "grouped_gemm")
    return out


def tile_gemm_supported(n: int, k: int, silu_mul: bool = False) -> bool:
    return k % 64 == 0 and n % 8 == 0 and (not silu_mul or (n // 2) % 32 == 0) and n * k * 2 < 2 ** 32


def tile_gemm(a, w, offsets=None, rows=None, arow_idx=None, silu_mul=False, residual=None, out=None, glu_clamp=None,
              relu_sq=False, xielu=None, gelu_mul=False, row_scale=None, parts=None):
    """The prefill GEMM (``csrc/kernels/tile_gemm.hip``): out[r] = epilogue(a[arow_idx[r] or r] @ w[g]^T).

    a [*, K] bf16; w [N, K] (dense) or [G, N, K] (grouped, with offsets [G + 1] int32 ON THE DEVICE:
    group g owns output rows offsets[g] .. offsets[g+1], no host synchronisation).  silu_mul: w is
    [gate rows | up rows], out = silu(gate) * up, [rows, N / 2].  residual [rows, N]: out = product +
    residual (``out`` may be ``residual`` itself).  glu_clamp = (limit, alpha, bias): w is [gate rows | up
    rows] as for silu_mul, out = min(g, limit) * sigmoid(alpha min(g, limit)) * (clamp(u, +-limit) + bias).
    relu_sq: out = relu(product)^2.  xielu = (a_pos, a_neg): out = a_pos z^2 + z / 2 for z > 0, else
    a_neg (exp(z) - 1 - z) + z / 2.  gelu_mul: paired like silu_mul, out = gelu(gate) * up with gelu in its tanh
    form.  row_scale (fp32 [rows], with glu_clamp): gate and up of an output row are multiplied by its factor before
    the clamps.  Rows at or past offsets[G] are left unwritten.  ``parts``: the workspace (``tail_parts``) of a caller that closes the
    tail's split tiles itself; dense products are closed here."""
    paired = silu_mul or glu_clamp is not None or gelu_mul
    if w.dim() == 2:
        w = w.unsqueeze(0)
    g, n, k = w.shape
    if rows is None:
        rows = a.shape[0] if arow_idx is None else arow_idx.numel()
    n_out = n // 2 if paired else n
    _bf16_cuda(a, w, residual)
    assert w.is_contiguous() and a.stride(-1) == 1 and a.shape[1] == k
    assert row_scale is None or (glu_clamp is not None and row_scale.is_cuda and row_scale.dtype == torch.float32
                                 and row_scale.is_contiguous() and row_scale.numel() >= rows)
    assert sum((silu_mul, glu_clamp is not None, relu_sq, residual is not None, xielu is not None, gelu_mul)) <= 1
    if offsets is not None:
        assert offsets.dtype == torch.int32 and offsets.numel() == g + 1 and offsets.is_cuda
    else:
        assert g == 1
    if arow_idx is not None:
        assert arow_idx.dtype == torch.int32 and arow_idx.is_cuda and arow_idx.numel() >= rows
    if out is None:
        out = torch.empty((rows, n_out), dtype=a.dtype, device=a.device)
    assert out.stride(-1) == 1 and out.shape[0] >= rows and out.shape[1] == n_out
    if residual is not None:
        assert residual.stride(-1) == 1 and residual.shape[0] >= rows and residual.shape[1] == n_out
    epi = 1 if silu_mul else 2 if residual is not None else 3 if glu_clamp is not None else 4 if relu_sq else 0
    lim, alpha, bias = glu_clamp if glu_clamp is not None else (0.0, 1.0, 0.0)
    if xielu is not None:
        epi, alpha, bias = 5, float(xielu[0]), float(xielu[1])
    if gelu_mul:
        epi = 6
    ws = parts
    if ws is None and offsets is None and epi <= 2 and _tail_pass_pays(rows, n, k, paired):
        ws = tail_parts(a.device, _tail_slots(rows, n, k, paired))
    rc = _kernels().vpsa_tile_gemm(_p(a), c_long(a.stride(0)), _p(arow_idx), _p(w), _p(offsets), c_int(g), _p(out),
                                   c_long(out.stride(0)), c_int(rows), c_int(n), c_int(k), c_int(epi), _p(residual),
                                   c_long(residual.stride(0) if residual is not None else 0), c_long(a.shape[0]),
                                   c_float(lim), c_float(alpha), c_float(bias), _p(row_scale), _p(ws), _stream())
    _check(rc, "tile_gemm")
    if ws is not None and parts is None:
        _tail_finish(ws, out, rows, n, k, epi, residual)
    return out


def _tiles(rows: int, n: int, paired: bool) -> int:
    return -(-rows // 256) * (-(-(n // 2) // 128) if paired else -(-n // 256))


def tile_tail(rows: int, n: int, k: int, paired: bool = False) -> int:
    """Ranges of the reduction that the last tiles of a dense product are cut in (1: none is), ``csrc/kernels/tile_tail.h``."""
    return int(_kernels().vpsa_tile_tail(c_int(_tiles(rows, n, paired)), c_int(k)))


TAIL_MIN_CHUNKS = 23  # the shortest reduction that saves 16 chunks in ranges of six or more


def _tail_pass_pays(rows: int, n: int, k: int, paired: bool) -> bool:
    """Whether a dense product's tail is cut, given the pass of its own that closes it: 5 to 10 us for the launch and little else while the
    ranges are few, twice that where they fill a round and their sums take 64 MB.  A tail alone then has to save 22 chunks: whole / cut,
    microseconds, 16384 x 2048 gated, 300 rows, 16 saved 38.5 / 44; x 2304, 18 saved 42.8 / 47; x 2560, 20 saved 53.2 / 51.9; 4096 x 2560
    residual, 2048 rows, 20 saved 59.0 / 59.8; 4096 x 1792, 1024 rows, 21 saved 38.2 / 40.0; 10880 x 2048, 500 rows, 22 saved 48.0 / 45.2."""
    splits, tiles, chunks = tile_tail(rows, n, k, paired), _tiles(rows, n, paired), k // 64
    return splits > 1 and (tiles >= TILE_CUS or tiles * splits <= 224 or chunks - chunks // splits >= 22)


def _tail_slots(rows: int, n: int, k: int, paired: bool) -> int:
    """Ranges of tail tiles that a dense product has in all."""
    return _tiles(rows, n, paired) % TILE_CUS * tile_tail(rows, n, k, paired)


def tail_parts(device, slots: int = TILE_CUS):
    """Room for the partial sums of that many tail workgroups, a tile of 256 x 256 each; a round of them is the most there is."""
    return torch.empty(slots << 16, dtype=torch.float32, device=device)


def _tail_finish(ws, out, rows, n, k, epi, residual):
    rc = _kernels().vpsa_tile_tail_finish(_p(ws), _p(out), c_long(out.stride(0)), c_int(rows), c_int(n), c_int(k), c_int(epi), _p(residual),
                                          c_long(0 if residual is None else residual.stride(0)), _stream())
    _check(rc, "tile_tail_finish")


def grouped_gemm_supported(n: int, k: int, silu_mul: bool = False) -> bool:
    return k % 64 == 0 and (not silu_mul or (n // 2) % 32 == 0)


def moe_experts_prefill(x, w13, w2, ids, weights, gather=True, foreign=False, combine=True):
    """Expert MLP for prefill-sized batches: the (token, k) pairs are sorted by expert on the device
    and two grouped matrix-core GEMMs run over all experts at once: gate_up gathers its token
    rows by index and fuses silu(gate) * up, down writes the sorted rows that the weighted combine
    gathers back; split tiles of the last product's tail are summed there too.  Four launches, no host synchronisation."""
    t, k = ids.shape
    if not x.is_cuda:
        return reference.moe_experts(x, w13, w2, ids, weights)
    n_experts = w13.shape[0]
    offsets, pos, sorted_tok = moe_align(ids, n_experts + (1 if foreign else 0))
    if foreign:  # the bucket of pairs held elsewhere ends the list: the GEMMs stop at offsets[n_experts]
        offsets = offsets[: n_experts + 1]
    gg = tile_gemm if (tile_gemm_supported(w13.shape[1], w13.shape[2], True)
                       and tile_gemm_supported(w2.shape[1], w2.shape[2])) else grouped_gemm
    if gather:
        act = gg(x, w13, offsets, rows=t * k, arow_idx=sorted_tok, silu_mul=True)
    else:  # copy the rows into sorted order first (timing comparison)
        act = gg(moe_permute(x, sorted_tok), w13, offsets, rows=t * k, silu_mul=True)
    # (from eight rounds of tiles on there is no tail, and none of short reductions whatever the routing (tile_tail.h); the host knows the
    # least number of tiles that a routing can make.  A thread finds each pair's place: 256 a token.)
    if (not combine or gg is not tile_gemm or -(-t * k // 256) * -(-w2.shape[1] // 256) >= 8 * TILE_CUS or w2.shape[2] < 64 * TAIL_MIN_CHUNKS
            or w2.shape[1] % 8 or k > 256 or t == 0):
        y = gg(act, w2, offsets, rows=t * k)
        if not combine:  # the caller sums the pairs itself
            return y, pos
        return moe_combine(y, weights, pos, t)
    tiles = (t * k // 256 + n_experts) * -(-w2.shape[1] // 256)  # the most that a routing makes
    ws = tail_parts(x.device, min(TILE_CUS, tiles * (w2.shape[2] // 64 // 6)))
    y = tile_gemm(act, w2, offsets, rows=t * k, parts=ws)
    assert weights.dtype == torch.float32 and pos.dtype == torch.int32
    out = torch.empty((t, w2.shape[1]), dtype=x.dtype, device=x.device)
    rc = _kernels().vpsa_moe_combine_parts(_p(ws), _p(offsets), c_int(n_experts), c_int(t * k), c_int(w2.shape[2]), _p(y),
                                           _p(weights.contiguous()), _p(pos), _p(out), c_int(t), c_int(w2.shape[1]), c_int(k), _stream())
    _check(rc, "moe_combine_parts")
    return out


def moe_experts_small_batch(x, w13, w2, ids, weights):
    """Expert MLP for a handful of tokens (decode): out[t] = sum_k weights[t,k] * MLP_{ids[t,k]}(x[t]).

    x [T, H] bf16, w13 [E, 2I, H] (gate rows then up rows), w2 [E, H, I], ids [T, K] int32,
    weights [T, K] fp32.  On the GPU only the routed experts' weights are streamed (two GEMV
    kernels + the weighted combine); no host synchronisation, HIP-graph capturable."""
    t, k = ids.shape
    if not x.is_cuda:
        return reference.moe_experts(x, w13, w2, ids, weights)
    _bf16_cuda(x, w13, w2)
    hidden, inter = x.shape[1], w2.shape[2]
    assert w13.shape[1] == 2 * inter and w13.shape[2] == hidden and w2.shape[1] == hidden
    assert w13.is_contiguous() and w2.is_contiguous() and ids.dtype == torch.int32
    act = torch.empty((t * k, inter), dtype=x.dtype, device=x.device)
    y = torch.empty((t * k, hidden), dtype=x.dtype, device=x.device)
    rc = _kernels().vpsa_moe_gemv(_p(x.contiguous()), _p(w13), _p(w2), _p(ids.contiguous()), _p(act), _p(y),
                                  c_int(t), c_int(k), c_int(hidden), c_int(inter), _stream())
    _check(rc, "moe_gemv")
    pos = torch.arange(t * k, dtype=torch.int32, device=x.device)
    return moe_combine(y, weights, pos, t)


# ---------------------------------------------------------------------------- LoRA
def lora_shrink(x, a, slots, rank_total):
    """h[t] = A[slots[t]] @ x[t] for rows with slots[t] >= 0 (other rows are left unwritten).

    x [T, in] bf16, a [S, R, in] bf16 (R = stacked, padded ranks), slots [T] int32 -> h [T, R] bf16."""
    t = x.shape[0]
    if not x.is_cuda:
        return reference.lora_shrink(x, a, slots)
    _bf16_cuda(x, a)
    assert a.is_contiguous() and a.shape[1] == rank_total and a.shape[2] == x.shape[1]
    assert slots.dtype == torch.int32 and slots.numel() == t and x.stride(1) == 1
    h = torch.empty((t, rank_total), dtype=x.dtype, device=x.device)
    rc = _kernels().vpsa_lora_shrink(_p(x), c_long(x.stride(0)), _p(a), _p(slots), _p(h), c_int(t),
                                     c_int(x.shape[1]), c_int(rank_total), c_int(a.shape[0]), _stream())
    _check(rc, "lora_shrink")
    return h


def lora_expand(h, bs, slots, y, r_pad):
    """For each sub-module i (the parts of a fused projection, side by side in y and in h):
    y[t, off_i : off_i + out_i] += B_i[slots[t]] @ h[t, i * r_pad : (i + 1) * r_pad], slots[t] >= 0.

    h [T, n * r_pad] bf16, bs: list of [S, out_i, r_pad] bf16 (adapter scale folded in),
    y [T, >= sum(out_i)] bf16, updated in place by one launch."""
    if not h.is_cuda:
        off = 0
        for i, b in enumerate(bs):
            reference.lora_expand(h, i * r_pad, b, slots, y, off)
            off += b.shape[1]
        return y
    _bf16_cuda(h, y, *bs)
    assert h.is_contiguous() and y.stride(1) == 1 and 1 <= len(bs) <= 3
    n = len(bs)
    outs = [b.shape[1] for b in bs]
    assert all(b.is_contiguous() and b.shape[2] == r_pad for b in bs) and sum(outs) <= y.shape[1]
    y_offs = [sum(outs[:i]) for i in range(n)]
    ptrs = (c_void_p * n)(*[b.data_ptr() for b in bs])
    rc = _kernels().vpsa_lora_expand(_p(h), c_int(h.stride(0)), ptrs, (c_int * n)(*outs),
                                     (c_int * n)(*y_offs), (c_int * n)(*[i * r_pad for i in range(n)]),
                                     c_int(n), _p(slots), _p(y), c_long(y.stride(0)), c_int(h.shape[0]),
                                     c_int(r_pad), c_int(bs[0].shape[0]), _stream())
    _check(rc, "lora_expand")
    return y


# --------------------------------------------------------------------------- latent attention, group routing, fp32 residual
from .latent import (add_rms_norm, build_latent_tiles, embed_scale, gate_up_glu_clamp, gather_rows, glu_clamp,  # noqa: E402,F401
                     depth_mix_rms_norm, embed_rms_norm, moe_glu, poly_norm, soft_cap, up_poly_norm,
                     gate_up_act, gated_add_rms_norm, glu_act, rms_norm_add, route_softmax,
                     group_topk, latent_attention, moe_glu_grouped, moe_glu_grouped_supported, moe_units, moe_units_grouped, up_relu_sq,
                     latent_expanded_supported, latent_kv_write, latent_mfma_supported, moe_finish, relu_sq, rms_norm_rows, rope_pairs, sigmoid_gate)

# --------------------------------------------------------------------------- recurrent mixers, windowed attention, Dynamic Tanh
from .seqmix import (add_dyt_norm, build_gru_pieces, build_scan_pieces, mingru_scan, build_window_tiles, head_rms_norm, mix_heads, recurrent_scan, short_conv_qkv,  # noqa: E402,F401
                     diff_heads, gla_prepare, head_finish, mlstm_prepare, pool_blocks, prepared_scan, qk_norm_write, scan_state_cols,
                     up_xielu, window_attention, window_cache_elems, window_decode_splits, window_kv_write, window_mfma_supported, xielu)
