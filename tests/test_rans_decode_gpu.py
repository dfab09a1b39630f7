"""The entropy decoder where its loop, its staging and its reads of the sizes change their way."""

import numpy as np
import pytest
import torch

from vllm_production_stack_amd import ops
from vllm_production_stack_amd.ops import reference as ref

DEV = torch.device("cuda")


# steps: less than a run of 16, whole runs, a remainder; bytes of 64 streams: what a thread asks for at once (14336), more, up to what LDS
# holds (320 a stream), and beyond
@pytest.mark.gpu
@pytest.mark.parametrize("per_stream", [1, 15, 16, 17, 33, 250, 262, 360, 372])
@pytest.mark.parametrize("shift", [0, 1])  # sizes at 16 and at 2 bytes
def test_rans_decode_edges(per_stream, shift):
    spc, n_ctx = 512, 3
    g = torch.Generator().manual_seed(per_stream)
    n = n_ctx * spc * per_stream
    sym = torch.randint(-64, 64, (n,), generator=g).to(torch.int8)  # seven bits a symbol
    sym[-spc * per_stream:] = 5
    freq, states, sizes, coded = (torch.from_numpy(np.ascontiguousarray(a).reshape(-1)) for a in ref.rans_encode(sym.numpy(), n_ctx, spc))
    at = torch.zeros(sizes.numel() + 8, dtype=torch.int16, device=DEV)[shift:shift + sizes.numel()]
    at.copy_(sizes.view(torch.int16))
    got = ops.rans_decode(freq.view(torch.int16).to(DEV), states.view(torch.int32).to(DEV), at, coded.to(DEV), n, n_ctx, spc)
    assert torch.equal(got.cpu(), sym)


# as many workgroups as the chip holds at once, and one context more (two launches, a wave for 64 streams)
@pytest.mark.gpu
@pytest.mark.parametrize("n_ctx", [96, 97])
@pytest.mark.parametrize("per_stream", [1, 17, 372])
@pytest.mark.parametrize("shift", [0, 1])
def test_rans_decode_many_contexts(n_ctx, per_stream, shift):
    spc = 512
    g = torch.Generator(device=DEV).manual_seed(per_stream)
    sym = torch.randint(-64, 64, (n_ctx * spc * per_stream,), generator=g, device=DEV).to(torch.int8)
    sym[-spc * per_stream:] = 5
    freq, states, sizes, coded = ops.rans_encode(sym, n_ctx, spc)
    at = torch.zeros(sizes.numel() + 8, dtype=torch.int16, device=DEV)[shift:shift + sizes.numel()]
    at.copy_(sizes.view(torch.int16))
    assert torch.equal(ops.rans_decode(freq, states, at, coded, sym.numel(), n_ctx, spc), sym)
