"""Products of ``csrc/kernels/block_gemm.hip`` whose workgroups make several tiles, one behind the other, against 64 bits."""

from ctypes import c_int

import pytest
import torch

from vllm_production_stack_amd import ops

BF = torch.bfloat16
# two to four rounds of workgroups, the last one ragged; reductions of fewer chunks than the ring has places, of as many, one more and many;
# rows, columns and batches that end inside a tile
CASES = [(26, 1000, 136, 768, 3), (33, 1000, 72, 64, 3), (33, 1000, 72, 128, 3), (33, 1000, 72, 192, 1), (22, 1500, 392, 128, 1), (26, 1000, 136, 128, 2),
         (1, 20001, 520, 256, 2), (31, 1549, 200, 320, 3), (7, 1501, 776, 192, 2), (1, 32700, 264, 3072, 1), (1, 8066, 1440, 1536, 1), (1, 29525, 520, 256, 1),
         (1, 16500, 768, 3072, 1), (1, 16500, 256, 512, 3)]
EPILOGUES = [(False, False), (True, False), (False, True)]  # gelu, residual


def _product(b, t, n, k, parts, gelu, residual):
    """Rows, columns, reduction and weights of a case (a residual goes with one weight)."""
    return (b * t, n * parts, k, 1) if residual else (b * t, n, k, parts)


def test_cases_reach_every_tile_shape_by_several_tiles_a_workgroup():
    at = lambda c, e: ops._kernels().vpsa_block_gemm_shape(*map(c_int, (*_product(*c, *e), *e)))  # noqa: E731
    reached = {(at(c, e), e) for c in CASES for e in EPILOGUES}
    assert reached >= {(16 + shape, e) for shape in range(6) for e in EPILOGUES}
    assert any(shape < 16 for shape, _ in reached)  # too short a reduction


def _rand(*shape, std=1.0):
    return torch.randn(*shape, device="cuda", dtype=torch.float32).mul_(std).to(BF)


@pytest.mark.gpu
@pytest.mark.parametrize("b,t,n,k,parts", CASES)
@pytest.mark.parametrize("gelu,residual", EPILOGUES)
def test_several_tiles_a_workgroup(b, t, n, k, parts, gelu, residual):
    torch.manual_seed(b + t + n + k)
    _, n, _, parts = _product(b, t, n, k, parts, gelu, residual)
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
