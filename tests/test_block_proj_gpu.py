"""Projections of about a hundred to a few hundred rows (``block_gemm``): heights of a row tile, one and two of them, columns that end inside a
tile, one chunk and uneven ranges of the reduction, the sums that close it, and which sizes the dispatch hands over."""

from ctypes import c_int

import pytest
import torch

from vllm_production_stack_amd import ops

pytestmark = pytest.mark.gpu
DEV, BF = torch.device("cuda"), torch.bfloat16


def _inputs(m, n, k):
    g = torch.Generator(device=DEV).manual_seed(m + n + k)
    x = torch.randn(m, k + 8, generator=g, device=DEV).to(BF)[:, :k]   # rows of a wider tensor
    return x, (torch.randn(n, k, generator=g, device=DEV) * k ** -0.5).to(BF), torch.randn(n, generator=g, device=DEV).to(BF), g


@pytest.mark.parametrize("m", [1, 97, 128, 129, 160, 161, 193, 224, 225, 256, 257, 321, 512])
@pytest.mark.parametrize("n,k,kind", [(128, 64, ""), (200, 320, "bias"), (520, 1088, ""), (256, 2624, "bias"), (336, 320, "pair"), (272, 1088, "pair"),
                                      (128, 8704, "")])
def test_matches_float64(m, n, k, kind):
    x, w, b, _ = _inputs(m, n, k)
    b = b if kind == "bias" else None
    splits = int(ops._kernels().vpsa_block_proj_splits(c_int(m), c_int(n), c_int(k), c_int(kind == "pair")))
    assert splits >= 1 and (splits > 1) == (k > 64 * 11)               # six chunks a range and more
    got = ops._split_product(ops._kernels().vpsa_block_proj, x, w, b, kind == "pair", splits)
    want = x.double() @ w.double().t()
    if kind == "pair":
        want = torch.nn.functional.silu(want[:, :n // 2]) * want[:, n // 2:]
    elif b is not None:
        want = want + b.double()
    # sums in 32 bits, one rounding to 16: half a unit in the last place, 2^-9, of every value
    assert float(((got.double() - want).abs() - want.abs() * 2 ** -8 - 1e-5).max()) < 0


@pytest.mark.parametrize("m,n,k", [(129, 4096, 8192), (256, 4096, 8192), (300, 4096, 8192), (512, 4096, 8192), (200, 4096, 4096)])
def test_sum_with_residual_and_norm(m, n, k):
    """Blocks with one and two row tiles, and two blocks of 128 rows: the separate passes' roundings."""
    x, w, _, g = _inputs(m, n, k)
    res, ln = torch.randn(m, n, generator=g, device=DEV).to(BF), torch.randn(n, generator=g, device=DEV).to(BF)
    got_res = res.clone()
    got = ops.block_add_norm(x, w, got_res, ln, 1e-5)
    assert got is not None
    add = x.double() @ w.double().t()
    want = add + res.double()
    # two roundings to 16 bits, of the sum and of the new row: half a unit in the last place, 2^-9, of each and the first's share again
    assert float(((got_res.double() - want).abs() - 2 ** -8 * (add.abs() + want.abs()) - 1e-5).max()) < 0
    norm = got_res.double() * (got_res.double().square().mean(1, keepdim=True) + 1e-5).rsqrt() * ln.double()
    assert float(((got.double() - norm).abs() - 2 ** -8 * norm.abs() - 1e-5).max()) < 0


@pytest.mark.parametrize("m", [129, 200, 256])
def test_sum_with_rotation_and_cache_write(m):
    n_q, n_kv, k = 32, 8, 4096
    x, w, b, g = _inputs(m, (n_q + 2 * n_kv) * 128, k)
    pool = torch.randn(m + 2, 2, 2, n_kv * 64 * 128, generator=g, device=DEV).to(BF)
    positions = torch.randint(0, 500, (m,), generator=g, device=DEV, dtype=torch.int32)
    slots = torch.randperm((m + 2) * 64, generator=g, device=DEV)[:m]
    slots[m // 2] = -1
    ang = torch.rand(500, 64, generator=g, device=DEV) * 6.28
    cos_sin = torch.cat([ang.cos(), ang.sin()], dim=1).contiguous()
    splits = ops._block_takes(x, w, b, False, ops.BLOCK_SUMS_QKV)
    want_pool, qkv = pool.clone(), ops._split_product(ops._kernels().vpsa_block_proj, x, w, b, False, splits)
    ops.rope_and_cache(qkv, positions, slots, cos_sin, want_pool, 1, n_q, n_kv, 128)
    q = ops.decode_qkv(x, w, b, pool, 1, positions, slots, cos_sin, n_q, n_kv)
    assert torch.equal(q, qkv[:, :n_q * 128]) and torch.equal(pool, want_pool)


def test_dispatch():
    def rule(m, n, k, pair=False, sums=ops.MID_SUMS):
        return ops._block_splits(m, n, k, pair, sums)

    assert rule(96, 28672, 4096, True) == 0 and rule(97, 28672, 4096, True) == 1 and rule(256, 28672, 4096, True) == 1
    assert rule(257, 28672, 4096, True) == 0                            # unsplit products of two row tiles
    assert rule(256, 57344, 8192, True) == 0 and rule(200, 57344, 8192, True) == 1    # a second round that is three quarters full
    assert rule(128, 4096, 14336) == 0 and rule(129, 4096, 14336) == 8 and rule(512, 4096, 14336) == 4 and rule(513, 4096, 14336) == 0
    assert rule(128, 8192, 28672) == 4                                  # beyond mid_gemm's weights
    assert rule(150, 6144, 4096) == 5 and rule(200, 6144, 4096) == 0 and rule(200, 6144, 4096, sums=ops.BLOCK_SUMS_QKV) == 5
    assert rule(129, 2048, 2048) == 0
    x, w, _, _ = _inputs(130, 28672, 512)
    assert ops._block_takes(x, w, None, True) == 1
    assert ops._block_takes(x.float(), w, None, True) == 0 and ops._block_takes(x, w.cpu(), None, True) == 0
    with torch.enable_grad():
        assert ops._block_takes(x.clone().requires_grad_(), w, None, True) == 0
