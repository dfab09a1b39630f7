"""Dense attention whose keys end inside a tile: what lies behind the last key in memory is not looked at."""

import pytest
import torch

from vllm_production_stack_amd import ops

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("tk", [1, 7, 8, 31, 32, 33, 40, 63, 64, 65, 96, 97, 128, 129, 191, 200])
@pytest.mark.parametrize("tq", [1, 130])
def test_keys_behind_the_last_one(tq, tk):
    torch.manual_seed(tk + tq)
    b, heads, c = 2, 3, 192
    q = torch.randn(b, tq, c, device="cuda").bfloat16()
    kv = torch.full((b, 2 * tk + 260, 2 * c + 64), float("nan"), device="cuda").bfloat16()  # rows of one tensor, every second, NaN elsewhere
    kv[:, : 2 * tk : 2, : 2 * c] = torch.randn(b, tk, 2 * c, device="cuda").bfloat16()
    k, v = kv[:, : 2 * tk : 2, :c], kv[:, : 2 * tk : 2, c : 2 * c]
    assert ops.dense_attention_supported(q, k, v, heads)
    got = ops.dense_attention(q, k, v, heads).double()
    qh, kh, vh = (x.double().view(b, -1, heads, 64).transpose(1, 2) for x in (q, k, v))
    p = torch.softmax(qh @ kh.transpose(-1, -2) * 0.125, -1)
    want, size = ((p @ x).transpose(1, 2).reshape(b, tq, c) for x in (vh, vh.abs()))
    # weights and result in 16 bits, eight of them significand: 2^-8 of every weight, so of the sum of absolute values, and of the result
    assert bool(((got - want).abs() <= 2 ** -8 * want.abs() + 1.05 * 2 ** -8 * size + 1e-5).all())
