"""The merge of a prompt tile's key ranges reads its records in runs of eight, four, two and one: every remainder, against the unsplit
reference."""

import math

import pytest
import torch

from test_kernels_gpu import BF, DEV, REL_TOL, _block_tables, _rel_row_err, _v_offset_pool
from vllm_production_stack_amd import ops
from vllm_production_stack_amd.ops import reference as ref

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("ranges", [2, 3, 5, 7, 8, 9, 12, 15, 17])
def test_any_number_of_ranges(ranges):
    n_q, n_kv, hd, rows_of, each = 8, 2, 128, 40, 4
    ctx = ranges * each * ops.PAGE - 5
    torch.manual_seed(ranges)
    pool = _v_offset_pool(ranges * each + 3, 1, n_kv, seed=ranges)
    bt = _block_tables(1, ranges * each, pool.shape[0], ranges)
    q = torch.randn(rows_of, n_q * hd, device=DEV).to(BF)
    i32 = lambda v: torch.tensor(v, dtype=torch.int32, device=DEV)  # noqa: E731
    cu, ctx_t, scale = i32([0, rows_of]), i32([ctx]), 1.0 / math.sqrt(hd)
    assert ops.prefill_tile_rows([rows_of], n_q, n_kv) == 64
    split = [v for i in range(ranges) for v in (i * each, (i + 1) * each, i)]
    ws = torch.full((ranges * ops.prefill_split_record_bytes(n_q, n_kv) // 4,), float("nan"), device=DEV)
    out = torch.zeros_like(q)
    ops.paged_prefill(q, out, pool, 0, bt, cu, ctx_t, i32([0] * ranges), i32([0] * ranges), n_q, n_kv, hd, scale, 64,
                      split=i32(split), split_ws=ws, groups=i32([0, 0, 0, ranges]))
    want = torch.zeros_like(q)
    ref.paged_prefill(q, want, pool, 0, bt, cu, ctx_t, n_q, n_kv, hd, scale)
    assert _rel_row_err(out, want, n_q) < REL_TOL


@pytest.mark.parametrize("ranges", [10, 31, 32, 33, 57])
def test_maxima_behind_the_first_eight_records(ranges):
    """Read beside the first run's values, 24 at a time: one such run, a whole one and one more, a third."""
    test_any_number_of_ranges(ranges)
