"""A page's parts and coded bytes straight into pinned memory, against the coder's own tensors."""

import pytest
import torch

from vllm_production_stack_amd import ops
from vllm_production_stack_amd.kv.serde import PageSerde, _Pinned

DEV = torch.device("cuda")


# groups of no byte, of less than a piece of 16, and of many pieces; what reaches the host ends anywhere, also between two groups' bytes
@pytest.mark.gpu
@pytest.mark.parametrize("spc,per_stream,spread", [(256, 1, 3), (256, 3, 1), (256, 40, 0), (512, 257, 40), (512, 256, 7)])
@pytest.mark.parametrize("head_bytes", [0, 16, 48000])
def test_publish_is_the_coders_output(spc, per_stream, spread, head_bytes):
    n_ctx = 3
    g = torch.Generator(device=DEV).manual_seed(per_stream)
    sym = torch.randint(-spread, spread + 1, (n_ctx * spc * per_stream,), generator=g, device=DEV).to(torch.int8)
    assert ops.rans_publishes(sym.numel(), n_ctx, spc)
    freq, states, sizes, coded = ops.rans_encode(sym, n_ctx, spc)
    head = torch.randint(0, 256, (head_bytes,), generator=g, device=DEV, dtype=torch.uint8)
    want = torch.cat([head, coded]).cpu()
    for cap in sorted({0, 5, head_bytes + coded.numel() // 2, head_bytes + coded.numel() // 2 + 7, want.numel() - 1, want.numel(), want.numel() + 100}):
        f, st, sz = torch.empty_like(freq), torch.empty_like(states), torch.empty_like(sizes)
        buf = torch.full((64 + max(cap, 16) + 64,), 77, dtype=torch.uint8).pin_memory()
        meta = torch.zeros(2, dtype=torch.int64).pin_memory()
        to = buf[64:64 + cap]
        if cap:
            ops.rans_encode_into(sym, n_ctx, f, st, sz, None, spc, meta=meta, page=(head, to))
        else:
            ops.rans_encode_into(sym, n_ctx, f, st, sz, None, spc, meta=meta, page=(head, buf[64:64]))
        torch.cuda.synchronize()
        assert meta.tolist() == [coded.numel(), 0]
        assert torch.equal(f, freq) and torch.equal(st, states) and torch.equal(sz, sizes)
        reach = min(cap, want.numel())
        if cap >= head_bytes:
            assert torch.equal(to[:reach], want[:reach])
        assert (buf[:64] == 77).all() and (buf[64 + reach:] == 77).all()


@pytest.mark.gpu
def test_a_page_that_its_buffer_does_not_hold():
    g = torch.Generator(device=DEV).manual_seed(5)
    serde = PageSerde(4, 8, 128, torch.bfloat16, "cachegen", levels=[127] * 4)
    page = torch.randn(serde.page_elems, generator=g, device=DEV).bfloat16()
    want = serde.encode(page)
    small = _Pinned(4096)
    serde._out_bufs.clear()
    serde._take, taken = (lambda bufs, size, _real=serde._take: taken.append(size) or (small if len(taken) == 1 else _real(bufs, size))), []
    assert serde.encode(page) == want and len(taken) == 2 and taken[1] > 4096
