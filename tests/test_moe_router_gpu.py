"""The router's product and the choice of experts (``csrc/kernels/moe.hip``) against 64 bits."""

import pytest
import torch

from vllm_production_stack_amd import ops
from vllm_production_stack_amd.ops import reference

pytestmark = pytest.mark.gpu
BF = torch.bfloat16


@pytest.mark.parametrize("tokens", [1, 15, 16, 17, 1531])
@pytest.mark.parametrize("experts,hidden", [(1, 128), (8, 4096), (16, 256), (17, 1152), (33, 640), (64, 2048)])
def test_router(tokens, experts, hidden, monkeypatch):
    monkeypatch.setattr(ops, "MOE_ROUTER_WEIGHTS", 1 << 30)  # (where the library is the better choice as well)
    monkeypatch.setattr(ops, "MOE_ROUTER_TOKENS", 1 << 30)
    torch.manual_seed(tokens + experts)
    x = torch.randn(tokens, hidden + 8, device="cuda").to(BF)[:, :hidden]
    w = (torch.randn(experts, hidden, device="cuda") * hidden ** -0.5).to(BF)
    want = x.double() @ w.double().t()
    err = (ops.moe_router(x, w).double() - want).abs()
    # one rounding to 16 bits, and sums of `hidden` products in 32
    assert bool((err <= want.abs() * 2 ** -8 + 1e-6).all()), err.max().item()


@pytest.mark.parametrize("experts,topk", [(2, 1), (8, 2), (8, 8), (9, 3), (16, 4), (31, 8), (60, 6), (64, 8)])
@pytest.mark.parametrize("tokens", [1, 7, 33, 1000])
def test_choice(tokens, experts, topk):
    torch.manual_seed(tokens + experts)
    logits = (torch.randn(tokens, experts, device="cuda") * 2).round().to(BF)  # many ties: the lowest expert first
    for renorm in (True, False):
        w, ids = ops.moe_topk_softmax(logits, topk, renorm)
        p = torch.softmax(logits.double(), dim=-1)
        order = torch.argsort(-logits.double(), dim=-1, stable=True)[:, :topk]
        want = p.gather(1, order)
        want = want / want.sum(-1, keepdim=True) if renorm else want
        assert torch.equal(ids.long(), order)
        assert float((w.double() - want).abs().max()) < 2e-6  # 32-bit exponentials (two units in the last place) and sums


def test_scores_that_are_no_numbers():
    nan, inf = float("nan"), float("inf")
    logits = torch.tensor([[1.0, nan, 3.0, 2.0], [nan, nan, nan, nan], [-inf, 0.0, -inf, -inf]], device="cuda").to(BF)
    w, ids = ops.moe_topk_softmax(logits, 2)
    assert ids[0].tolist() == [2, 3] and ids[1].tolist() == [0, 0] and ids[2].tolist() == [1, 0]
    assert w[0].isnan().all() and w[1].isnan().all() and w[2].tolist() == [1.0, 0.0]
