"""What the products refuse, on the host and in front of any launch. Needs no GPU."""

from ctypes import c_float, c_int, c_void_p

import pytest
import torch

from qwen3_runtime_amd.ops.hip import HipOps, OpsError


# scaled rows are a residual's, of up to 4,096 columns; few rows of more asked for 64 KB of LDS beside the factors and were refused by the launch
@pytest.mark.parametrize("m,k", [(9, 4160), (16, 4160), (1, 8192), (17, 2560), (4, 96)])
@pytest.mark.parametrize("gated,shared", [(-1, 0), (0, 0), (0, 1)])
def test_scaled_products_take_rows_of_a_residual(m, k, gated, shared):
    lib = HipOps().lib
    somewhere = c_void_p(1 << 20)  # not read: the sizes are refused
    code = lib.qrt_scaled_gemm_bf16(somewhere, somewhere, somewhere, c_int(m), c_int(12304), c_int(k), c_int(gated), c_float(0.0), c_int(shared),
                                    somewhere, c_float(1e-6), None)
    assert code != 0 and f"bad sizes M={m} N=12304 K={k}" in lib.qrt_last_error().decode()


# where the gate went by a pass of its own, the rotated columns were left as they were
@pytest.mark.parametrize("dtype", [torch.bfloat16, torch.float32])
def test_products_per_head_take_a_gate_or_a_rotation(dtype):
    x, w, out = torch.zeros(2, 4 * 64, dtype=dtype), torch.zeros(4, 64, 64, dtype=dtype), torch.zeros(2, 4 * 96, dtype=dtype)
    rotation = dict(in_stride=64, in_offset=32, out_stride=96, out_offset=64, heads=4, width=32, positions=torch.zeros(2, dtype=torch.int32),
                    freq=torch.ones(16))
    with pytest.raises(OpsError, match="not both"):
        HipOps().heads_linear(x, 64, 0, w, out, 96, 0, gate=torch.zeros_like(out), rotation=rotation)
