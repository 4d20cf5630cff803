"""Which tiles float32 products take: the choice beside what the three of them were measured to take, and a product by each."""

from ctypes import c_int

import pytest
import torch

from test_float32_ring_gpu import check
from test_kernels_gpu import rnd

from qwen3_runtime_amd.ops.hip import HipOps, _ptr, _stream

TILES = (64064, 64032, 32032)


# us by 64 x 64, 64 x 32 and 32 x 32 (csrc/gemm_f32.hip): two runs of one product differ by 2 to 3 %
@pytest.mark.parametrize("n,k,planes,times", [
    (19456, 2560, 0, {65: (152, 139, 110), 128: (133, 118, 117), 192: (172, 175, 178), 354: (331, 318, 316), 400: (383, 373, 358), 512: (416, 402, 412),
                      1024: (791, 833, 941), 2048: (1542, 1684, 1691)}),
    (6144, 2560, 0, {128: (66, 51, 42), 230: (96, 75, 76), 354: (131, 118, 105), 512: (131, 133, 136), 1024: (258, 276, 308), 2048: (496, 533, 541)}),
    (2560, 9728, 4, {128: (88, 66, 60), 354: (160, 162, 159), 512: (209, 202, 208), 1024: (400, 420, 468), 2048: (768, 842, 857)}),
    (12288, 4096, 0, {448: (405, 382, 406), 700: (607, 589, 643)}),
    (13824, 5120, 0, {900: (1069, 1131, 1226)}),
])
def test_the_tile_is_the_fastest_or_next_to_it(n, k, planes, times):
    lib = HipOps().lib
    for rows, us in times.items():
        assert us[TILES.index(lib.qrt_gemm_f32_tile_of(rows, n, k, planes))] <= 1.035 * min(us), (rows, us)


# 64 x 64 tiles in whole rounds of the compute units and a remainder of either side; k: one stage, a last part that ends early, 16 parts
@pytest.mark.gpu
@pytest.mark.parametrize("m,n", [(1983, 4033), (1955, 4035)])
@pytest.mark.parametrize("k", [32, 288, 1056, 8224])
def test_whole_product_by_square_tiles(m, n, k):
    ops = HipOps(residual_planes=True)
    assert ops.lib.qrt_gemm_f32_tile_of(m, n, k, 0) == 64064
    x, w = rnd(m, k, seed=5), rnd(n, k, seed=6, scale=0.05)
    check(ops.linear(x, w), x, w, lambda rows: ops.linear(rows, w))


# blocks that are alone on their units, with weights that lie in L2 from the pass before: through registers (us through them and by the ring 10.3 and 12.4,
# 6.5 and 7.5, 18.3 and 24.3); short K, larger weights, more blocks than units, four planes of them: by the ring
@pytest.mark.parametrize("m,n,k,planes,ring", [(65, 1024, 1024, 0, 0), (300, 256, 512, 0, 0), (300, 16, 2048, 0, 0), (65, 256, 768, 4, 0),
                                               (65, 1024, 96, 0, 1), (65, 2048, 2048, 0, 1), (300, 1024, 1024, 0, 1), (300, 256, 768, 4, 1),
                                               (300, 2048, 2050, 0, 0)])
def test_what_goes_through_the_ring(m, n, k, planes, ring):
    assert HipOps().lib.qrt_gemm_f32_ring_of(m, n, k, planes) == ring


# sums of groups: four and seven blocks to a unit (two slots in the ring), five and six (three), remainders of either side
@pytest.mark.gpu
@pytest.mark.parametrize("m,n", [(2041, 1987), (2041, 3267), (2049, 1987), (2049, 2563)])
@pytest.mark.parametrize("k", [256, 288, 1056, 8224])
def test_sums_of_groups_by_square_tiles(m, n, k):
    ops = HipOps(residual_planes=True)
    x, w = rnd(m, k, seed=7), rnd(n, k, seed=8, scale=0.05)

    def product(rows, planes):
        out = torch.full((planes, rows.shape[0], n), float("nan"), device=x.device)
        ops._check(ops.lib, ops.lib.qrt_gemm_f32_planes(_ptr(rows), _ptr(w), _ptr(out), c_int(rows.shape[0]), c_int(n), c_int(k), c_int(planes), _stream()))
        return out[0] if planes == 1 else ((out[0] + out[1]) + out[2]) + out[3]

    check(product(x, 1), x, w, lambda rows: product(rows, 4))
