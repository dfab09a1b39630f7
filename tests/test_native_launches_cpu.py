"""A launch that the runtime refuses is an error of the call, not a result that nobody wrote.  (Where there is no GPU every launch is refused.)"""

from ctypes import c_float, c_int, c_long, c_void_p

import pytest
import torch

from vllm_production_stack_amd import ops

pytestmark = pytest.mark.skipif(torch.cuda.is_available(), reason="launches are refused where there is no GPU")
AT = c_void_p(4096)  # no launch, so nothing reads there
CALLS = {
    "vpsa_rans_decode": (AT, c_long(64), AT, AT, AT, None, AT, c_long(2 * 512 * 4), c_int(2), c_int(512)),
    "vpsa_row_add": (AT, c_long(64), AT, AT, AT, AT, AT, c_int(3), c_int(128), c_int(64)),
    "vpsa_row_qkv": (AT, c_long(64), AT, c_float(1e-5), AT, AT, AT, c_int(3), c_int(64), AT, AT, AT, AT, c_long(64), c_long(64), c_int(2), c_int(1)),
    "vpsa_mid_unit_factors": (AT, c_long(512), AT, c_float(1e-5), AT, AT, c_long(16384), c_int(3), c_int(32768), c_int(512)),
    "vpsa_mid_gemm": (AT, c_long(4096), AT, None, AT, c_long(28672), None, c_int(3), c_int(28672), c_int(4096), c_int(0), c_int(1)),
    "vpsa_dense_attention": (4096, 64, 64, 4096, 4096, 64, 64, 4096, 64, 64, 1, 3, 70, 1, 0.125),
}


@pytest.mark.parametrize("entry", CALLS)
def test_a_refused_launch_is_an_error(entry):
    assert getattr(ops._kernels(), entry)(*CALLS[entry], None) not in (0, -1)  # (-1: the call's own checks)
