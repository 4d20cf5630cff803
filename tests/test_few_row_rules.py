"""Which kernel takes few rows: both sides of the lines that were measured."""

import pytest

from qwen3_runtime_amd.ops.hip import HipOps


# evenly shared rows (csrc/gemm_even.h), us by tiles and evenly: 5,120 x 64 at 16 rows 2.8, 2.9; 8,200 x 4,096 at 1 row 13.6, 16.0; 11,264 x 6,144 at 8 rows 9 % apart; 10,240 x 6,144
# at 1 row 23.6, 25.0
@pytest.mark.parametrize("m,n,k,evenly", [
    (1, 6144, 2560, 1), (8, 10240, 2560, 1), (16, 9728, 4096, 1), (1, 6144, 640, 1), (8, 12288, 2560, 1), (16, 10304, 1024, 1), (1, 4160, 4096, 1), (1, 8320, 8192, 1),
    (1, 8200, 2560, 1), (9, 11264, 5120, 1), (8, 10240, 6144, 1), (1, 6144, 8192, 1),
    (16, 5120, 64, 0), (9, 9000, 192, 0), (12, 12000, 320, 0), (9, 4104, 1024, 0), (1, 8200, 4096, 0), (8, 8256, 8192, 0), (5, 12288, 4096, 0), (7, 12288, 2560, 0),
    (8, 11264, 6144, 0), (16, 12288, 960, 0), (8, 4096, 2560, 0), (8, 7168, 2560, 0), (8, 12289, 2560, 0), (7, 10240, 6144, 0), (1, 6144, 12288, 0),
])
def test_rows_that_are_shared_evenly(m, n, k, evenly):
    assert HipOps().lib.qrt_gemm_even_takes(m, n, k) == evenly
