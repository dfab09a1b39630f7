"""KV pages that come in on a stream of their own: many in a row without a wait, on other streams and threads than the default, beside
other work in the memory that they were given, against the same pages one at a time."""

import ctypes
import threading
from collections import deque

import pytest
import torch

from vllm_production_stack_amd import ops
from vllm_production_stack_amd.kv.serde import PageSerde, _Pinned

pytestmark = pytest.mark.gpu
DEV, BF = torch.device("cuda"), torch.bfloat16


@pytest.fixture(scope="module", params=[(4, 8), (32, 8)], ids=["below 2 MB", "above"])
def pages(request):
    layers, n_kv = request.param
    serde = PageSerde(layers, n_kv, 128, BF, "cachegen")
    g = torch.Generator(device=DEV).manual_seed(layers)
    blobs = [serde.encode(torch.randn(serde.page_elems, generator=g, device=DEV).to(BF)) for _ in range(5)]
    assert (len(blobs[0]) > 2 << 20) == (layers == 32)
    want = []
    for b in blobs:
        want.append(PageSerde(layers, n_kv, 128, BF, "cachegen").decode(b, DEV))
        torch.cuda.synchronize()
    return serde, blobs, want


def test_in_a_row(pages):
    serde, blobs, want = pages
    for _ in range(3):
        got = []
        for b in blobs:
            got.append(serde.decode(b, DEV))
            torch.empty(1 << 23, dtype=torch.uint8, device=DEV).fill_(255)   # memory that a page's workspace has just left
        assert all(torch.equal(x, y) for x, y in zip(got, want))


def test_streams_and_threads(pages):
    serde, blobs, want = pages
    got = {}

    def call(i):
        s = torch.cuda.Stream()
        with torch.cuda.stream(s):
            for rep in range(4):
                got[i, rep] = serde.decode(blobs[(i + rep) % 5], DEV).clone()
        s.synchronize()

    threads = [threading.Thread(target=call, args=(i,)) for i in range(4)]
    for t in threads:
        t.start()
    for t in threads:
        t.join(60)
    assert len(got) == 16 and all(torch.equal(y, want[(i + rep) % 5]) for (i, rep), y in got.items())


def test_behind_work_that_is_still_queued(pages):
    """A buffer that is new lies where the stream's queued work still writes."""
    serde, blobs, want = pages
    fresh = PageSerde(serde.n_layers, serde.n_kv, 128, BF, "cachegen")
    a = torch.randn(4096, 4096, device=DEV)
    for _ in range(4):
        a = a @ a * 1e-3
        torch.empty(len(blobs[0]) + len(blobs[0]) // 8, dtype=torch.uint8, device=DEV).fill_(7)
    assert torch.equal(fresh.decode(blobs[1], DEV), want[1])


def test_no_stream_that_others_are_handed(pages):
    """torch's pool deals its streams out in turn: whoever gets one may capture on it."""
    lib = ops._kernels()
    lib.vpsa_page_copy_stream.restype = ctypes.c_void_p
    own = lib.vpsa_page_copy_stream()
    assert own and own == lib.vpsa_page_copy_stream()
    assert own not in {torch.cuda.Stream().cuda_stream for _ in range(100)}


def test_a_new_buffer_holds_up_no_other_stream(pages):
    """A page that comes in behind a stream's queued work with a buffer that is new; then one on another stream, with one that is not.  (Streams share
    a few hardware queues, so not every pair is independent; where every page waits for the one before, none is.)"""
    serde, blobs, want = pages
    a = torch.randn(8192, 8192, device=DEV).to(BF)
    out, free, streams = torch.empty_like(a), 0, [torch.cuda.Stream() for _ in range(6)]

    def new():
        s = PageSerde(serde.n_layers, serde.n_kv, 128, BF, "cachegen")
        s._in_bufs = deque([_Pinned(2 * len(blobs[1]))])  # (kept when the call is over: whoever drops a buffer waits for its copy)
        return s

    for s in streams:
        with torch.cuda.stream(s):
            new().decode(blobs[0], DEV), serde.decode(blobs[0], DEV), torch.mm(a, a, out=out)
    for i in range(6):
        torch.cuda.synchronize()
        busy, other, fresh = streams[i], streams[(i + 1) % 6], new()
        with torch.cuda.stream(busy):
            for _ in range(100):
                torch.mm(a, a, out=out)
            late = fresh.decode(blobs[1], DEV)
            passed = torch.cuda.Event()
            passed.record()
        with torch.cuda.stream(other):
            got = serde.decode(blobs[2], DEV)
            other.synchronize()
        free += not passed.query()
        assert torch.equal(got, want[2])
        busy.synchronize()
        assert torch.equal(late, want[1])
    assert free > 0
