"""float32 products whose K is whole stages of 32, which come through a ring of direct loads, at the edges of their tiles: float64
within the bound of a float32 sum, and the bits of few rows (another kernel)."""

import pytest
import torch

from test_kernels_gpu import DEV, rnd

pytestmark = pytest.mark.gpu


@pytest.fixture(scope="module")
def ops():
    from qwen3_runtime_amd.ops.hip import HipOps

    return HipOps(residual_planes=True)


def check(whole, x, w, few):
    bound = x.shape[1] * 2.0 ** -24 * (x.double().abs() @ w.double().abs().T)   # k products in any order, each rounded
    assert ((whole.double() - x.double() @ w.double().T).abs() <= bound).all()
    for first, m in ((0, 1), (63, 9), (whole.shape[0] - 32, 32)):
        assert torch.equal(few(x[first: first + m].contiguous()), whole[first: first + m]), (first, m)


# m, n: 32 x 32, 64 x 32 and 64 x 64 tiles with remainders of both (columns past the last group of four too), one tile in all, tiles no multiple
# of the eight XCDs; k: one stage, one a part, a last part that ends early, no stage in the last parts, an odd number, 16 parts
@pytest.mark.parametrize("m,n", [(97, 1), (97, 131), (301, 2561), (301, 6148), (2049, 4097)])
@pytest.mark.parametrize("k", [32, 64, 96, 288, 1056, 8224])
def test_whole_product(ops, m, n, k):
    x, w = rnd(m, k, seed=1), rnd(n, k, seed=2, scale=0.05)
    check(ops.linear(x, w), x, w, lambda rows: ops.linear(rows, w))


# in planes by every tile, and as their sum; k: groups of two parts of which the last has none, of one stage a part, an odd number, of four
@pytest.mark.parametrize("m,n", [(97, 65), (200, 2562), (520, 2562), (2049, 2563)])
@pytest.mark.parametrize("k", [256, 288, 1056, 8224])
def test_product_for_the_residual(ops, m, n, k):
    x, w = rnd(m, k, seed=3), rnd(n, k, seed=4, scale=0.05)
    added = lambda p: p if p.dim() == 2 else ((p[0] + p[1]) + p[2]) + p[3]
    whole, few = ops.linear_for_residual(x, w), ops.linear_for_residual(x[:32].contiguous(), w)
    if whole.dim() == few.dim():
        assert torch.equal(whole[..., :32, :], few)
    check(added(whole), x, w, lambda rows: added(ops.linear_for_residual(rows, w)))
