"""Which kernel takes few rows: both sides of the lines that were measured."""

import pytest

import test_gated_rows_gpu as gated

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


# gated rows by five waves (csrc/gemm_bf16.hip), us by three and five at 64 rows: 9,728 x 128 5.8, 7.3; 2,048 x 768 11 % apart; 9,728 x 2,048 5 %; 5,120 x 768 2 %
@pytest.mark.parametrize("n,k,five", [
    (256, 1536, 1), (1536, 1536, 1), (2048, 2560, 1), (4352, 1024, 1), (6144, 2048, 1), (9728, 2560, 1), (10240, 5120, 1),
    (256, 1024, 0), (1536, 1472, 0), (1552, 1536, 0), (2048, 2304, 0), (5120, 768, 0), (9728, 128, 0), (9728, 2048, 0), (3072, 4096, 0), (12288, 4096, 0),
])
def test_gated_rows_by_five_waves(n, k, five):
    assert HipOps().lib.qrt_gated_gemm_mixed(n, k) == five


# rows: ends of the blocks of 16; outputs: fewer tiles than compute units, one tile to some of three, five to all; K: two k-steps less than a chunk of ten,
# whole chunks, a chunk and a part
@pytest.mark.gpu
@pytest.mark.parametrize("m", [9, 16, 17, 48, 49, 64])
@pytest.mark.parametrize("n,k", [(48, 1536), (48, 1600), (1536, 1664), (4112, 1088), (10240, 2560), (10240, 2624)])
def test_gated_products_by_five_waves(m, n, k):
    assert HipOps().lib.qrt_gated_gemm_mixed(n, k) == 1
    gated.test_gated_rows(m, n, k)
