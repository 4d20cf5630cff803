"""What the products refuse, on the host and in front of any launch. Needs no GPU."""

from ctypes import c_float, c_int, c_void_p

import pytest

from qwen3_runtime_amd.ops.hip import HipOps


# scaled rows are a residual's, of up to 4,096 columns; few rows of more asked for 64 KB of LDS beside the factors and were refused by the launch
@pytest.mark.parametrize("m,k", [(9, 4160), (16, 4160), (1, 8192), (17, 2560), (4, 96)])
@pytest.mark.parametrize("gated,shared", [(-1, 0), (0, 0), (0, 1)])
def test_scaled_products_take_rows_of_a_residual(m, k, gated, shared):
    lib = HipOps().lib
    somewhere = c_void_p(1 << 20)  # not read: the sizes are refused
    code = lib.qrt_scaled_gemm_bf16(somewhere, somewhere, somewhere, c_int(m), c_int(12304), c_int(k), c_int(gated), c_float(0.0), c_int(shared),
                                    somewhere, c_float(1e-6), None)
    assert code != 0 and f"bad sizes M={m} N=12304 K={k}" in lib.qrt_last_error().decode()
