"""Products of ``csrc/kernels/block_gemm.hip`` whose workgroups make several tiles, one behind the other, against 64 bits."""

import pytest
import torch

from vllm_production_stack_amd import ops

pytestmark = pytest.mark.gpu
BF = torch.bfloat16


def _rand(*shape, std=1.0):
    return torch.randn(*shape, device="cuda", dtype=torch.float32).mul_(std).to(BF)


# two to four rounds of workgroups, the last one ragged; reductions of fewer chunks than the ring has places, of as many, one more and many;
# each tile shape that such products choose; rows, columns and batches that end inside a tile
@pytest.mark.parametrize("b,t,n,k,parts", [(26, 1000, 136, 768, 3), (33, 1000, 72, 64, 3), (33, 1000, 72, 128, 3), (33, 1000, 72, 192, 1),
                                           (22, 1500, 392, 128, 1), (26, 1000, 136, 128, 2), (1, 20001, 520, 256, 2), (31, 1549, 200, 320, 3),
                                           (7, 1501, 776, 192, 2)])
@pytest.mark.parametrize("gelu,residual", [(False, False), (True, False), (False, True)])
def test_several_tiles_a_workgroup(b, t, n, k, parts, gelu, residual):
    torch.manual_seed(b + t + n + k)
    if residual:  # (one weight only)
        n, parts = n * parts, 1
    x, ws = _rand(b, t + 1, k)[:, :t], [_rand(n, k, std=k ** -0.5) for _ in range(parts)]
    biases, res = [_rand(n) if p != 1 else None for p in range(parts)], _rand(b, t, n * parts) if residual else None
    buf = torch.full((b, t + 3, n * parts), 7.0, dtype=BF, device="cuda")
    assert ops.block_linear(x, ws, biases, gelu, residual=res, out=buf[:, 1 : t + 1]) is not None
    for i in range(b):
        y = torch.cat([x[i].double() @ w.double().t() + (0 if v is None else v.double()) for w, v in zip(ws, biases)], dim=-1)
        want = (torch.nn.functional.gelu(y) if gelu else y) + (res[i].double() if residual else 0)
        # one rounding to 16 bits, and 32-bit sums of k products: 2^-8 of the value and a part of the sum's size
        err = (buf[i, 1 : t + 1].double() - want).abs()
        assert bool((err <= want.abs() * 2 ** -8 + 1e-6 * k ** 0.5).all()), err.max().item()
    assert bool((buf[:, 0] == 7).all()) and bool((buf[:, t + 1 :] == 7).all())
