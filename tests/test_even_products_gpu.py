"""Few rows by weights whose rows are shared out evenly over the compute units (csrc/gemm_even.hip), against float64."""

import pytest
import torch

pytestmark = pytest.mark.gpu
DEV = "cuda:0"
EPS = 1e-6


@pytest.fixture(scope="module")
def ops():
    from qwen3_runtime_amd.ops.hip import HipOps

    return HipOps(residual_planes=True)


def rnd(*shape, seed, scale=1.0, dtype=torch.bfloat16):
    g = torch.Generator().manual_seed(seed)
    return (torch.randn(*shape, generator=g) * scale).to(dtype).to(DEV)


# columns: 16 and 17 rows a block (in some blocks the third unit has no row), 24, 32 and 33, 40, 40 and 41, 48, and just outside of what is shared
# evenly; K: one pair of k-steps, fewer pairs than waves, one more than fills their rings, many
@pytest.mark.parametrize("m", [1, 4, 5, 8, 9, 16])
@pytest.mark.parametrize("n", [4096, 4104, 4368, 6144, 6160, 8192, 8200, 10240, 10248, 12288, 12304])
def test_whole_products(ops, m, n):
    for k in (64, 192, 832, 2560):
        x, w = rnd(m, k, seed=1), rnd(n, k, seed=2, scale=k ** -0.5)
        want = x.double() @ w.double().T
        # K additions in float32 of products that are exact there, and the result's rounding to bfloat16
        bound = (x.double().abs() @ w.double().abs().T) * (k + 16) * 2.0 ** -24 + want.abs() * 2.0 ** -8
        assert ((ops.linear(x, w).double() - want).abs() <= bound).all(), k
        # the same sums, in the float32 result that goes by tiles: the same bits
        assert torch.equal(ops.linear(x, w), ops.linear(x, w, out_f32=True).to(torch.bfloat16)), k
        if n % 16 == 0:
            assert torch.equal(ops.act_linear(x, w, "relu2"), ops.unary_act(ops.linear(x, w), "relu2")), k


@pytest.mark.parametrize("m", [1, 5, 8, 9, 16])
@pytest.mark.parametrize("n", [4112, 6144, 8208, 10240, 12288])
@pytest.mark.parametrize("k", [256, 2560])
def test_rows_that_lack_their_norms_factor(ops, m, n, k):
    residual, x = rnd(m, k, seed=1, dtype=torch.float32), rnd(m, 512, seed=2)
    w, weight, wider = rnd(k, 512, seed=3, scale=0.05), 1.0 + 0.1 * rnd(k, seed=4, dtype=torch.float32), rnd(n, k, seed=5, scale=k ** -0.5)
    stream = residual.double() + x.double() @ w.double().T
    normed = stream / torch.sqrt(stream.square().mean(-1, keepdim=True) + EPS) * weight.double()
    sums, size = normed @ wider.double().T, normed.abs() @ wider.double().abs().T
    rows = ops.add_rmsnorm(residual, ops.product_for_norm(x, w), weight, EPS, torch.bfloat16, scaled=True)
    assert type(rows).__name__ == "ScaledRows"
    # one rounding of the rows and one of the result to bfloat16 (2^-9 each), and the sums' own
    allowed = size * (2.0 ** -9 + (k + 64) * 2.0 ** -23) + sums.abs() * 2.0 ** -8
    assert ((ops.linear(rows, wider).double() - sums).abs() <= allowed).all()
