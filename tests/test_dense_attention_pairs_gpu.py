"""Dense attention where pairs of waves share rows: few workgroups, and what is left behind whole rounds of 1024."""

import pytest
import torch

from vllm_production_stack_amd import ops

pytestmark = pytest.mark.gpu


def check(q, k, v, heads):
    b, tq, tk = q.shape[0], q.shape[1], k.shape[1]
    assert ops.dense_attention_supported(q, k, v, heads)
    got = ops.dense_attention(q, k, v, heads).double()
    qh, kh, vh = (x.double().view(b, -1, heads, 64).transpose(1, 2) for x in (q, k, v))
    p = torch.softmax(qh @ kh.transpose(-1, -2).contiguous() * 0.125, -1)
    want, size = ((p @ x).transpose(1, 2).reshape(b, tq, heads * 64) for x in (vh, vh.abs()))
    # weights and result in 16 bits, eight of them significand: half a unit is up to 2^-8 of every weight, so of the sum of absolute values,
    # and of the result; scores and sums are kept in 32
    assert bool(((got - want).abs() <= 2 ** -8 * want.abs() + 1.05 * 2 ** -8 * size + 1e-5).all())


@pytest.mark.parametrize("tk", [64, 65, 127, 128, 129, 191, 192, 193, 257])  # one tile (by itself), an odd and an even number, each end
@pytest.mark.parametrize("b,heads,tq", [(1, 1, 1), (2, 3, 63), (1, 8, 64), (1, 9, 65), (2, 4, 193), (4, 8, 1000), (33, 1, 1000)])
def test_few_workgroups(b, heads, tq, tk):  # 8 to 256 blocks of 128 rows, and 320 that are not cut
    torch.manual_seed(tk + tq)
    q, kv = torch.randn(b, tq, heads * 64, device="cuda").bfloat16(), torch.randn(b, tk, heads * 128 + 8, device="cuda").bfloat16()
    check(q, kv[..., : heads * 64], kv[..., heads * 64 : heads * 128], heads)


@pytest.mark.parametrize("b,tq", [(127, 1000), (128, 1000), (129, 1000), (144, 1020), (145, 1000), (257, 1000)])
def test_what_is_left_behind_rounds(b, tq):  # 1016 to 1160 blocks and 2048 + 64: none left, 64 (with idle ones), 128, 192 (not cut)
    torch.manual_seed(b)
    q, k, v = (torch.randn(b, t, 64, device="cuda").bfloat16() for t in (tq, 200, 200))
    check(q, k, v, 1)


@pytest.mark.parametrize("first", [0, 64])
def test_one_wave_of_a_pair_has_all_the_weight(first):
    """Keys of every other tile far below the others, and without a score at all: their wave's sums count for nothing."""
    torch.manual_seed(first)
    q, k, v = (torch.randn(1, t, 64, device="cuda").bfloat16() for t in (100, 300, 300))
    q[..., 0] = 8.0
    low = (torch.arange(300, device="cuda") // 64 % 2 == 1) == (first == 0)
    for score in (-1000.0, float("-inf")):
        k[:, low, 0] = score
        check(q, k, v, 1)


@pytest.mark.parametrize("tk", [128, 192, 320, 448])  # whole tiles: no key past the last one is read in its place
@pytest.mark.parametrize("at", [0, 100, -1])
def test_values_without_bound(tk, at):
    torch.manual_seed(tk)
    q, k, v = (torch.randn(2, t, 64, device="cuda").bfloat16() for t in (70, tk, tk))
    v[0, at, 3], v[0, at, 40], v[1, at, 7] = float("inf"), float("-inf"), float("nan")
    want = torch.softmax(q.double() @ k.double().transpose(-1, -2).contiguous() * 0.125, -1) @ v.double()
    got = ops.dense_attention(q, k, v, 1).double()
    assert torch.equal(got.isnan(), want.isnan()) and torch.equal(got[got.isinf()], want[want.isinf()]) and torch.equal(got.isinf(), want.isinf())
    bound = want.isfinite()
    assert float((got - want)[bound].norm() / want[bound].norm()) < 2 ** -7
