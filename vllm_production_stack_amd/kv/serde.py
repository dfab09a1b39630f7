"""KV page serialisation for the disk and remote tiers.

``naive``    header + raw page bytes (what every reference example configures:
             /root/reference/tutorials/assets/values-06-shared-storage.yaml:53).
``cachegen`` lossy: anchor-delta + layer-dependent quantisation on the GPU
             (``cachegen_encode`` kernel), then an entropy stage.  On a GPU that stage is the
             interleaved rANS coder of ``csrc/kernels/rans.hip`` (serde kind 2: the page is
             quantised, coded and packed on the device, the compressed bytes are what crosses
             PCIe; decoding mirrors it).  On a CPU-only host it is the adaptive range coder of
             ``libvpsa_kvio`` (kind 1, ~30 M symbols/s).  Both are 2-4x smaller than bf16; either
             side reads both kinds.

Wire format: 32-byte header ``VPKV | version u16 | serde u16 | n_layers u32 | n_kv u32 |
head_dim u32 | page_tokens u32 | payload_len u64`` followed by the payload.  For cachegen
the payload is ``scales fp32[n_groups] | rc_len u64 | range-coded symbols`` (kind 1) or
``spc u32 | streams u32 | coded_len u64 | scales fp32[n_groups] | freq u16[n_layers * 256] |
states u32[streams] | sizes u16[streams] | coded bytes`` (kind 2).
"""

from __future__ import annotations

import ctypes
import os
import struct
from collections import deque

import numpy as np
import torch

from .. import _native, ops

MAGIC = b"VPKV"
SERDE_NAIVE, SERDE_CACHEGEN = 0, 1
# quantiser + GPU rANS entropy stage (what a GPU engine writes for "cachegen"); kind 1, the
# host range coder, remains for CPU hosts and for blobs already stored
SERDE_CACHEGEN_RANS = 2
_RANS_HDR = struct.Struct("<IIQ")  # streams per context, streams, coded bytes
_KEPT = 2  # pinned buffers a serialiser keeps for each direction
_HDR = struct.Struct("<4sHHIIIIQ")

# a bytes object made at its size and filled before anyone else sees it (the C API's way to build one without a second copy)
_new_bytes = ctypes.PYFUNCTYPE(ctypes.py_object, ctypes.c_void_p, ctypes.c_ssize_t)(("PyBytes_FromStringAndSize", ctypes.pythonapi))
_bytes_at = ctypes.PYFUNCTYPE(ctypes.c_void_p, ctypes.py_object)(("PyBytes_AsString", ctypes.pythonapi))

_kvio = None


def kvio():
    global _kvio
    if _kvio is None:
        lib = _native.load("vpsa_kvio")
        lib.kvio_rc_encode.restype = ctypes.c_int64
        lib.kvio_rc_encode.argtypes = [ctypes.c_void_p, ctypes.c_size_t, ctypes.c_void_p,
                                       ctypes.c_size_t, ctypes.c_size_t, ctypes.c_int]
        lib.kvio_rc_decode.restype = ctypes.c_int
        lib.kvio_rc_decode.argtypes = [ctypes.c_void_p, ctypes.c_size_t, ctypes.c_void_p,
                                       ctypes.c_size_t, ctypes.c_size_t, ctypes.c_int]
        _kvio = lib
    return _kvio


def rc_encode(symbols: np.ndarray, ctx_period: int, n_ctx: int) -> bytes:
    symbols = np.ascontiguousarray(symbols, dtype=np.int8)
    cap = symbols.size + symbols.size // 8 + 64
    out = np.empty(cap, dtype=np.uint8)
    n = kvio().kvio_rc_encode(symbols.ctypes.data, symbols.size, out.ctypes.data, cap, ctx_period, n_ctx)
    if n < 0:
        raise RuntimeError("range coder output buffer too small")
    return out[:n].tobytes()


def rc_decode(data: bytes, n: int, ctx_period: int, n_ctx: int) -> np.ndarray:
    buf = np.frombuffer(data, dtype=np.uint8)
    out = np.empty(n, dtype=np.int8)
    if kvio().kvio_rc_decode(buf.ctypes.data, buf.size, out.ctypes.data, n, ctx_period, n_ctx) != 0:
        raise ValueError("range-coded KV payload is truncated or corrupt")
    return out


def default_levels(n_layers: int) -> list[int]:
    """Quantisation levels per layer: early layers are the most sensitive to KV error and
    keep 8 bits; the last two thirds step down to ~6 and ~5 bits."""
    a, b = n_layers // 3, 2 * n_layers // 3
    return [127 if i < a else (31 if i < b else 15) for i in range(n_layers)]


class _Pinned:
    """A pinned buffer on its way through a call, and what the device still has to pass before the buffer's memory may be used again.
    Its copies are queued by the kernel library, so torch's allocator knows nothing of them: whoever lets go of the buffer waits."""

    __slots__ = ("bytes", "busy")

    def __init__(self, size: int):
        self.bytes = torch.empty(size, dtype=torch.uint8, pin_memory=True)
        self.busy = None  # a stream or an event: over with its ``synchronize``

    def wait(self) -> None:
        if self.busy is not None:
            self.busy.synchronize()
            self.busy = None

    def __del__(self):
        if getattr(self, "busy", None) is not None:
            self.wait()


class PageSerde:
    def __init__(self, n_layers: int, n_kv: int, head_dim: int, dtype: torch.dtype, kind: str = "naive",
                 levels: list[int] | None = None):
        self.n_layers, self.n_kv, self.head_dim, self.dtype = n_layers, n_kv, head_dim, dtype
        self.kind = SERDE_CACHEGEN if kind == "cachegen" else SERDE_NAIVE
        self.page_elems = n_layers * 2 * n_kv * ops.PAGE * head_dim
        self.unit_elems = n_kv * ops.PAGE * head_dim
        self.levels = levels or default_levels(n_layers)
        self._levels_dev: dict = {}
        # Pinned buffers that pages pass through on their way between host and device: a pageable copy of a page's 3.5 MB takes
        # 0.65 ms to the host and 0.13 ms to the device, a pinned one 0.07.  A call takes one out and gives it back, so calls of
        # several threads do not wait for each other; at most two of each kind are kept, which lets one thread copy a page in
        # while the one before is on its way.
        self._out_bufs: deque = deque()
        self._in_bufs: deque = deque([None] * _KEPT)

    def __getstate__(self):  # (pinned buffers and device tensors stay with the object they were made for)
        return {**self.__dict__, "_levels_dev": {}, "_out_bufs": deque(), "_in_bufs": deque([None] * _KEPT)}

    @staticmethod
    def _take(bufs: deque, size: int) -> _Pinned:
        """A pinned buffer of at least ``size`` bytes that no copy reads any more."""
        try:
            buf = bufs.popleft()
        except IndexError:
            buf = None
        if buf is not None:
            buf.wait()
        if buf is None or buf.bytes.numel() < size:
            buf = _Pinned(size + size // 8)
        return buf

    @staticmethod
    def _give(bufs: deque, buf: _Pinned) -> None:
        if len(bufs) < _KEPT:
            bufs.append(buf)

    def _header(self, payload_len: int) -> bytes:
        return _HDR.pack(MAGIC, 1, self.kind, self.n_layers, self.n_kv, self.head_dim, ops.PAGE,
                         payload_len)

    # ------------------------------------------------------------------ encode
    def encode(self, page: torch.Tensor) -> bytes:
        """``page``: one KV page (any device), ``page_elems`` elements."""
        flat = page.reshape(-1)
        if self.kind == SERDE_NAIVE or self.unit_elems % 8192 != 0 or flat.dtype != torch.bfloat16:
            raw = flat.contiguous().cpu().view(torch.uint8).numpy().tobytes()
            return _HDR.pack(MAGIC, 1, SERDE_NAIVE, self.n_layers, self.n_kv, self.head_dim, ops.PAGE,
                             len(raw)) + raw
        if self._rans_ok(flat.device):
            return self._rans_page(flat, self._new_blob)
        sym_np, sc_np = self.quantize(flat)
        return self.pack(sym_np, sc_np)

    def _rans_ok(self, device) -> bool:
        return (torch.device(device).type == "cuda" and (2 * self.unit_elems) % ops.RANS_SPC == 0
                and os.environ.get("VPSA_CACHEGEN_HOST_CODER", "0") != "1")

    def quantize(self, flat: torch.Tensor):
        """GPU half of the cachegen encoder.  On a GPU: anchor/delta quantisation kernel and the
        rANS entropy stage, one device-to-host copy of the finished payload -> (payload, None).
        Otherwise the int8 symbols and fp32 scales come back for the host range coder
        -> (symbols, scales)."""
        if self._rans_ok(flat.device):
            return self._rans_page(flat, self._new_payload), None
        sym, scales = ops.cachegen_encode(flat.contiguous(), self._levels(flat.device), self.unit_elems, self.n_layers)
        return sym.cpu().numpy(), scales.float().cpu().numpy()

    def _levels(self, device) -> torch.Tensor:
        lv = self._levels_dev.get(device)
        if lv is None:
            lv = self._levels_dev[device] = torch.tensor(self.levels, dtype=torch.int32, device=device)
        return lv

    def _new_blob(self, payload: int):
        """(a stored page with room for ``payload`` bytes behind its header, the payload's address)"""
        blob = _new_bytes(None, _HDR.size + payload)
        at = _bytes_at(blob)
        ctypes.memmove(at, self._rans_header(payload), _HDR.size)
        return blob, at + _HDR.size

    @staticmethod
    def _new_payload(payload: int):
        out = np.empty(payload, dtype=np.uint8)
        return out, out.ctypes.data

    def _rans_page(self, flat: torch.Tensor, new):
        """A page's kind-2 payload in what ``new`` makes for its size.  Every stage writes its part of the payload where it belongs,
        the last one the size into pinned memory; then the payload is copied to the host in parts, and out of the pinned buffer
        behind them."""
        n, dev, n_streams = flat.numel(), flat.device, self.n_layers * ops.RANS_SPC
        o1 = 4 * (n // 64)
        o2 = o1 + 512 * self.n_layers
        o3 = o2 + 4 * n_streams
        o4 = o3 + 2 * n_streams
        body = torch.empty(o4 + 2 * n, dtype=torch.uint8, device=dev)
        sym, _ = ops.cachegen_encode(flat.contiguous(), self._levels(dev), self.unit_elems, self.n_layers,
                                     scales=body[:o1].view(torch.float32))
        ops.ensure_device()
        stream = torch.cuda.current_stream()  # the one that the kernel library queues on
        buf = self._take(self._out_bufs, o4 + n)  # (a value rarely codes to more than a byte)
        buf.busy = stream
        meta = buf.bytes[:16].view(torch.int64)
        ops.rans_encode_into(sym.view(-1), self.n_layers, body[o1:o2], body[o2:o3], body[o3:o4], body[o4:], meta=meta)
        stream.synchronize()
        total, bad = meta.tolist()
        if bad:
            raise RuntimeError("rans_encode: frequency table could not be normalised")
        if buf.bytes.numel() < o4 + total:
            buf = self._take(self._out_bufs, o4 + total)
            buf.busy = stream
        done, at = new(_RANS_HDR.size + o4 + total)
        ctypes.memmove(at, _RANS_HDR.pack(ops.RANS_SPC, n_streams, total), _RANS_HDR.size)
        ops.fetch_bytes(body, buf.bytes, at + _RANS_HDR.size, o4 + total)
        buf.busy = None  # (fetched: nothing is queued behind it)
        self._give(self._out_bufs, buf)
        return done

    def rans_payload(self, sym: torch.Tensor, scales: torch.Tensor) -> np.ndarray:
        """The kind-2 payload of symbols that are quantised already, coded where they lie: on a CPU-only host the definition
        that ``encode``'s pages on a GPU are equal to."""
        freq, states, sizes, coded = ops.rans_encode(sym.view(-1), self.n_layers)
        body = torch.cat([scales.float().contiguous().view(-1).view(torch.uint8),
                          freq.view(torch.uint8), states.view(torch.uint8), sizes.view(torch.uint8), coded])
        head = _RANS_HDR.pack(ops.RANS_SPC, states.numel(), coded.numel())
        return np.concatenate([np.frombuffer(head, dtype=np.uint8), body.cpu().numpy()])

    def _rans_header(self, payload_len: int) -> bytes:
        return _HDR.pack(MAGIC, 1, SERDE_CACHEGEN_RANS, self.n_layers, self.n_kv, self.head_dim, ops.PAGE, payload_len)

    def pack(self, sym_np: np.ndarray, sc_np: np.ndarray | None) -> bytes:
        """Host half: frame a finished rANS payload, or range-code the symbols (releases the
        GIL: safe to run on worker threads)."""
        if sc_np is None:
            return b"".join((self._rans_header(sym_np.size), memoryview(np.ascontiguousarray(sym_np)).cast("B")))
        coded = rc_encode(sym_np, 2 * self.unit_elems, self.n_layers)
        payload = sc_np.tobytes() + struct.pack("<Q", len(coded)) + coded
        return self._header(len(payload)) + payload

    def uses_codec(self, page: torch.Tensor) -> bool:
        return (self.kind == SERDE_CACHEGEN and self.unit_elems % 8192 == 0
                and page.dtype == torch.bfloat16)

    # ------------------------------------------------------------------ decode
    def _open(self, blob: bytes):
        """Header checks shared by every decoder: (kind, payload).  Anything that is not a whole
        page blob of this model's geometry is a ``ValueError``: blobs come from disk and from
        other hosts, and a damaged one must read as a cache miss, never as a wrong page."""
        if len(blob) < _HDR.size:
            raise ValueError("not a KV page blob")
        magic, ver, kind, nl, nkv, hd, pt, plen = _HDR.unpack_from(blob, 0)
        if magic != MAGIC or ver != 1:
            raise ValueError("not a KV page blob")
        if (nl, nkv, hd, pt) != (self.n_layers, self.n_kv, self.head_dim, ops.PAGE):
            raise ValueError("KV page geometry mismatch")
        if plen != len(blob) - _HDR.size:
            raise ValueError("truncated KV page blob")
        payload = memoryview(blob)[_HDR.size:]
        if kind == SERDE_NAIVE:
            if plen != self.page_elems * torch.empty((), dtype=self.dtype).element_size():
                raise ValueError("KV page blob of the wrong size")
        elif kind == SERDE_CACHEGEN_RANS:
            if plen < _RANS_HDR.size:
                raise ValueError("damaged cachegen payload")
        elif kind == SERDE_CACHEGEN:
            if plen < 4 * (self.page_elems // 64) + 8:
                raise ValueError("damaged cachegen payload")
        else:
            raise ValueError(f"unknown KV page encoding {kind}")
        return kind, payload

    def decode(self, blob: bytes, device: torch.device) -> torch.Tensor:
        kind, payload = self._open(blob)
        if kind == SERDE_NAIVE:
            t = torch.frombuffer(bytearray(payload), dtype=torch.uint8).view(self.dtype)
            return t.to(device)
        if kind == SERDE_CACHEGEN_RANS:
            return self.restore_rans(np.frombuffer(payload, dtype=np.uint8), device)
        sym_np, sc_np = self._unpack_payload(payload)
        return self.dequantize(sym_np, sc_np, device)

    def restore_rans(self, payload: np.ndarray, device) -> torch.Tensor:
        """rANS payload (host bytes) -> KV page on ``device``: one host-to-device copy, entropy
        decode and dequantisation on the GPU (NumPy definitions on a CPU-only host)."""
        spc, n_streams, coded_len = _RANS_HDR.unpack_from(payload, 0)
        n, a = self.page_elems, _RANS_HDR.size
        o1 = 4 * (n // 64)
        o2 = o1 + 2 * 256 * self.n_layers
        o3 = o2 + 4 * n_streams
        o4 = o3 + 2 * n_streams
        size = o4 + coded_len
        if n_streams != self.n_layers * spc or a + size > payload.size:
            raise ValueError("damaged cachegen payload")
        body = payload[a:a + size]
        if torch.device(device).type == "cuda":
            body = np.ascontiguousarray(body)
            ops.ensure_device()
            stream = torch.cuda.current_stream()  # the one that the kernel library queues on
            buf = self._take(self._in_bufs, size)
            buf.busy = stream  # until there is an event, also if the call ends early
            out = ops.page_decode(body.ctypes.data, buf.bytes, size, n, self.n_layers, self.unit_elems, device, spc)
            buf.busy = torch.cuda.Event()
            buf.busy.record(stream)
            self._give(self._in_bufs, buf)
            return out
        body = torch.from_numpy(body.copy()).to(device)
        sym = ops.rans_decode(body[o1:o2].view(torch.int16), body[o2:o3].view(torch.int32), body[o3:o4].view(torch.int16), body[o4:],
                              n, self.n_layers, spc)
        return ops.cachegen_decode(sym, body[:o1].view(torch.float32), self.unit_elems)

    def restore(self, got: tuple, device) -> torch.Tensor:
        """Finish what ``unpack`` started (its "codec" and "rans" results)."""
        if got[0] == "rans":
            return self.restore_rans(got[1], device)
        return self.dequantize(got[1], got[2], device)

    def _unpack_payload(self, payload) -> tuple[np.ndarray, np.ndarray]:
        n_groups = self.page_elems // 64
        scales = np.frombuffer(payload[: 4 * n_groups], dtype=np.float32).copy()
        (clen,) = struct.unpack_from("<Q", payload, 4 * n_groups)
        if clen != len(payload) - 4 * n_groups - 8:
            raise ValueError("damaged cachegen payload")
        coded = bytes(payload[4 * n_groups + 8:])
        return rc_decode(coded, self.page_elems, 2 * self.unit_elems, self.n_layers), scales

    def unpack(self, blob: bytes):
        """Host half of decode for worker threads: ("raw", uint8 array) for a naive blob,
        ("codec", symbols, scales) for a cachegen one."""
        kind, payload = self._open(blob)
        if kind == SERDE_NAIVE:
            return ("raw", np.frombuffer(payload, dtype=np.uint8).copy())
        if kind == SERDE_CACHEGEN_RANS:
            return ("rans", np.frombuffer(payload, dtype=np.uint8))  # entropy decode happens on the GPU
        return ("codec",) + self._unpack_payload(payload)

    def dequantize(self, sym_np: np.ndarray, sc_np: np.ndarray, device: torch.device) -> torch.Tensor:
        sym = torch.from_numpy(sym_np)
        scales = torch.from_numpy(sc_np)
        return ops.cachegen_decode(sym.to(device), scales.to(device), self.unit_elems)
