"""Prefill GEMM tiles of one to four units of 64 rows (``csrc/kernels/tile_gemm.hip``), grouped and dense, against 64 bits."""

import pytest
import torch

from vllm_production_stack_amd import ops

pytestmark = pytest.mark.gpu
BF = torch.bfloat16


def _rand(*shape, std=1.0):
    return torch.randn(*shape, device="cuda", dtype=torch.float32).mul_(std).to(BF)


def _close(got, want, terms):
    """One rounding to 16 bits, and 32-bit sums of ``terms`` products: 2^-8 of the value and a part of the sum's size."""
    err = (got.double() - want).abs()
    assert bool((err <= want.abs() * 2 ** -8 + 1e-6 * terms ** 0.5).all()), err.max().item()


# groups a row below, at and above every unit, of one to six units and none at all
@pytest.mark.parametrize("sizes", [[1, 63, 64, 65], [127, 128, 0, 129], [191, 192, 193, 255], [256, 257, 320, 321], [383, 385, 449, 0, 2]])
@pytest.mark.parametrize("silu", [False, True])
def test_groups(sizes, silu):
    torch.manual_seed(sum(sizes))
    n, k, rows, g = 320, 192, sum(sizes), len(sizes)
    a, w = _rand(rows + 9, k), _rand(g, n, k, std=k ** -0.5)
    idx = torch.randperm(rows + 9, device="cuda")[:rows].int()
    offs = [sum(sizes[:i]) for i in range(g + 1)]
    got = ops.tile_gemm(a, w, torch.tensor(offs, dtype=torch.int32, device="cuda"), rows=rows, arow_idx=idx, silu_mul=silu)
    want = torch.cat([a[idx[lo:hi].long()].double() @ w[i].double().t() for i, (lo, hi) in enumerate(zip(offs, offs[1:]))])
    if silu:
        gate, up = want.chunk(2, dim=-1)
        want = torch.nn.functional.silu(gate) * up
    _close(got, want, k)


@pytest.mark.parametrize("m", [1, 64, 65, 192, 193, 256, 320, 450, 513, 700, 1000])
def test_dense_with_residual(m):
    torch.manual_seed(m)
    n, k = 264, 128
    x, w, r = _rand(m, k), _rand(n, k, std=k ** -0.5), _rand(m + 3, n)
    want = x.double() @ w.double().t() + r[:m].double()
    got = r.clone()
    ops.tile_gemm(x, w, residual=got[:m], out=got[:m])
    _close(got[:m], want, k)
    assert torch.equal(got[m:], r[m:])
