"""Rules of the native kernels that the host can be asked for: no GPU takes part."""

from ctypes import c_int, c_long

import pytest
import torch

from vllm_production_stack_amd import ops


# chunks of a product's reduction or of one of its ranges: rows of 4096, 3584, 2048, 3072, 6144 and ranges of eight and more chunks
@pytest.mark.parametrize("n", [8, 16, 24, 28, 32, 40, 48, 56, 64, 72, 96, 112, 120])
def test_workgroups_of_a_projection_begin_apart(n):
    def first(block):
        return ops._kernels().vpsa_mid_first_chunk(c_int(block), c_int(n), c_int(0))

    assert all(0 <= first(b) < n for b in range(512))
    assert len({first(b) for b in range(8)}) == 8                        # the XCDs (workgroups go round them)
    for xcd in range(8):                                                 # an XCD's, as many as there are CUs
        assert len({first(b) for b in range(xcd, 256, 8)}) >= min(32, n // (3 if n % 3 == 0 else 1))
    assert len({first(b) for b in range(256)}) >= 0.8 * n                # no part of the row that nobody begins with


@pytest.mark.parametrize("n", [1, 2, 7, 12, 13, 64, 128, 152, 224])
def test_workgroups_of_whole_products_begin_apart(n):
    starts = [ops._kernels().vpsa_mid_first_chunk(c_int(b), c_int(n), c_int(1)) for b in range(512)]
    assert all(0 <= s < n for s in starts) and len(set(starts)) >= n // (3 if n % 3 == 0 else 1)


def test_threads_that_share_a_copy():
    """A copy has a thread for every 640 KB, up to four: starting one costs more than copying less."""
    def parts(size):
        return ops._kernels().vpsa_copy_parts(c_long(size))

    kb = 1 << 10
    assert [parts(n) for n in (0, 1, 51 * kb, 640 * kb, 1280 * kb - 1)] == [1] * 5
    assert [parts(n) for n in (1280 * kb, 1920 * kb, 2560 * kb, 7 << 20, 1 << 40)] == [2, 3, 4, 4, 4]


def test_routers_that_the_kernel_takes():
    """Short rows, few experts and one round of workgroups: elsewhere the library is up to four times as fast."""
    takes = ops.moe_router_takes
    assert all(takes(t, e, h) for t in (1, 8, 1531, 4096) for e, h in ((2, 4096), (8, 4096), (16, 2048), (32, 1024), (60, 512), (64, 512)))
    assert not any(takes(8, e, h) for e, h in ((8, 6144), (9, 4096), (16, 4096), (32, 2048), (60, 2048), (64, 1024), (65, 128), (128, 128)))
    assert not takes(4097, 8, 4096) and not takes(8, 8, 4000)


@pytest.mark.parametrize("heads,kv_heads,hidden", [(64, 8, 8192), (32, 8, 4096), (32, 4, 8192), (28, 4, 3584)])
@pytest.mark.parametrize("rows", [1, 64, 96, 97, 112, 128, 129, 176, 256])
def test_projections_that_write_the_cache_take_the_kernel_that_they_take_by_themselves(monkeypatch, heads, kv_heads, hidden, rows):
    """Rotation and cache in the reduction are a launch less, no reason for the slower product."""
    lib, called = ops._kernels(), []

    class Recorder:
        def __getattr__(self, name):
            if name.endswith("_splits"):
                return getattr(lib, name)
            return lambda *args: called.append(name) or 0

    n = (heads + 2 * kv_heads) * 128
    x, w = torch.empty((rows, hidden), dtype=torch.bfloat16), torch.empty((n, hidden), dtype=torch.bfloat16)
    slots, positions = torch.empty(rows, dtype=torch.int64), torch.empty(rows, dtype=torch.int32)
    pool, cos_sin = torch.empty((2, 1, 2, kv_heads, 64 * 128), dtype=torch.bfloat16), torch.empty((64, 128))
    monkeypatch.setattr(ops, "_kernels", Recorder)
    monkeypatch.setattr(ops, "_reads", lambda *_: True)
    monkeypatch.setattr(ops, "_stream", lambda: None)
    with torch.no_grad():
        itself = ["vpsa_block_proj_qkv"] if ops._block_splits(rows, n, hidden, False) > 1 else ["vpsa_mid_gemm_qkv"] if ops._mid_splits(rows, n, hidden, False) > 1 else []
        ops.decode_qkv(x, w, None, pool, 0, positions, slots, cos_sin, heads, kv_heads)
    assert called == itself or (not itself and called == ["vpsa_block_proj_qkv"])  # (which may take more partial sums here)


def test_entropy_decoders_of_many_contexts_have_a_launch_for_their_tables():
    """What one round of workgroups holds is decoded in one launch without a workspace; a page that codes to more has room for the tables."""
    def sizes(n_ctx, per_stream):
        n = n_ctx * 512 * per_stream
        return [int(f(c_long(n), c_int(n_ctx), c_int(512))) for f in (ops._kernels().vpsa_rans_decode_workspace, ops._kernels().vpsa_page_workspace)]

    assert sizes(1, 4) == [0, 2048] and sizes(80, 256) == [0, 80 * 512 * 256] and sizes(96, 16) == [0, 96 * 512 * 16]
    for n_ctx in (97, 126, 2048):
        tables = n_ctx * (4096 * 4 + 8)
        assert sizes(n_ctx, 16) == [tables, n_ctx * 512 * 16 + tables]


# widths and rows, microseconds of a decode step of 6 layers with the split products / with those of a few rows on an MI355X
@pytest.mark.parametrize("hidden,rows,split,whole", [
    (5120, 4, 724.6, 731.0), (5120, 8, 747.0, 770.1), (5120, 14, 783.1, 851.8), (6144, 1, 923.2, 900.5), (6144, 8, 954.8, 953.3), (6144, 11, 980.0, 1000.2),
    (6144, 14, 991.3, 1032.1), (7168, 8, 975.3, 954.6), (7168, 11, 999.5, 1011.0), (7168, 14, 1012.2, 1048.0), (8192, 14, 1295.6, 1280.6), (4096, 14, 657.9, 634.7),
    (3584, 14, 605.7, 593.3), (3072, 14, 530.6, 511.0)])
def test_products_of_a_few_rows_are_taken_where_they_are_faster(hidden, rows, split, whole):
    assert (rows <= ops.row_limit(hidden)) == (whole < split)


# windows, heads, query rows, keys, microseconds with whole blocks of 128 rows / with blocks cut in two on an MI355X
@pytest.mark.parametrize("b,heads,tq,tk,whole,cut", [
    (1, 8, 1, 1500, 21.6, 13.9), (8, 8, 4, 1500, 21.8, 14.1), (1, 8, 64, 65, 4.80, 4.97), (2, 12, 64, 129, 5.60, 5.95), (3, 20, 4, 129, 5.23, 5.42), (3, 20, 64, 200, 6.49, 6.16),
    (1, 12, 130, 65, 5.41, 5.00), (1, 8, 500, 129, 6.21, 6.00), (8, 8, 130, 300, 7.94, 7.11), (4, 8, 500, 448, 9.60, 8.25), (1, 8, 1500, 1500, 23.0, 15.4),
    (1, 12, 1500, 129, 6.62, 7.55), (2, 8, 1500, 300, 8.22, 9.31), (1, 12, 1500, 700, 13.03, 13.62), (1, 12, 1500, 1000, 16.9, 15.9), (2, 8, 1500, 1500, 23.27, 22.29),
    (8, 8, 500, 129, 6.99, 7.77), (3, 20, 500, 448, 10.46, 11.32), (8, 8, 500, 1500, 24.31, 23.42), (8, 12, 1500, 1500, 84.2, 80.8), (22, 8, 1500, 1500, 140.3, 135.4)])
def test_attention_blocks_are_cut_where_that_is_faster(b, heads, tq, tk, whole, cut):
    left = ops._kernels().vpsa_dense_attention_cut(c_int(b), c_int(heads), c_int(tq), c_int(tk))
    assert (left > 0) == (cut < whole)
    assert ops._kernels().vpsa_dense_attention_cut(c_int(b), c_int(heads), c_int(tq), c_int(64)) == 0  # a single tile
    assert left <= -(-b * heads // 8) * 8 * -(-tq // 128) and left % 8 == 0
