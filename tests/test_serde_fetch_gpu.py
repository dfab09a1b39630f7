"""What a page's encoder leaves to the runtime's copy: a kernel that gathers a page in LDS and stores it into host memory keeps its places on the chip as
long as the link takes, and a step on another stream waits for them."""

import pytest
import torch

from vllm_production_stack_amd import ops
from vllm_production_stack_amd.kv.serde import PageSerde, _Pinned

pytestmark = pytest.mark.gpu
DEV = torch.device("cuda")


def _page(serde, seed):
    return torch.randn(serde.page_elems, generator=torch.Generator(device=DEV).manual_seed(seed), device=DEV).bfloat16()


@pytest.mark.parametrize("payload", [False, True])
def test_kernels_write_nothing_but_the_size_into_host_memory(monkeypatch, payload):
    serde = PageSerde(4, 8, 128, torch.bfloat16, "cachegen")
    page = _page(serde, 1)
    encode = (lambda: serde.quantize(page)[0].tobytes()) if payload else (lambda: serde.encode(page))
    want = encode()
    buf = _Pinned(2 * serde.page_elems)
    buf.bytes.fill_(77)
    serde._out_bufs.clear()
    serde._out_bufs.append(buf)
    real, seen = ops.fetch_bytes, []

    def fetch(src, pinned, dst, size):
        torch.cuda.synchronize()
        assert pinned.data_ptr() == buf.bytes.data_ptr() and src.is_cuda
        seen.append(int((pinned != 77).sum()))
        real(src, pinned, dst, size)

    monkeypatch.setattr(ops, "fetch_bytes", fetch)
    assert encode() == want
    assert len(seen) == 1 and seen[0] <= 16


def test_a_page_that_its_buffer_does_not_hold():
    serde = PageSerde(4, 8, 128, torch.bfloat16, "cachegen", levels=[127] * 4)
    page = _page(serde, 5)
    want = serde.encode(page)
    small = _Pinned(4096)
    serde._out_bufs.clear()
    serde._take, taken = (lambda bufs, size, _real=serde._take: taken.append(size) or (small if len(taken) == 1 else _real(bufs, size))), []
    assert serde.encode(page) == want and len(taken) == 2 and taken[1] > 4096
