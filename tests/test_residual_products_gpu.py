"""Few rows: the product that is added to the residual stream in its own kernel, and the products that read rows which lack
their norm's factor (csrc/gemm_residual.hip, csrc/gemm_bf16.hip), against the same in float64."""

import pytest
import torch

pytestmark = pytest.mark.gpu
DEV = "cuda:0"
EPS = 1e-6


@pytest.fixture(scope="module")
def ops():
    from qwen3_runtime_amd.ops.hip import HipOps

    return HipOps(residual_planes=True)


def rnd(*shape, seed, scale=1.0, dtype=torch.float32):
    g = torch.Generator().manual_seed(seed)
    return (torch.randn(*shape, generator=g) * scale).to(dtype).to(DEV)


def exact(residual, x, w, weight, wider):
    """In float64: the stream, the sums of the rows that a product reads by (``wider``: its weight), and the size of their addends."""
    stream = residual.double() + x.double() @ w.double().T
    normed = stream / torch.sqrt(stream.square().mean(-1, keepdim=True) + EPS) * weight.double()
    return stream, normed @ wider.double().T, normed.abs() @ wider.double().abs().T


# 8 and 16 rows: the ends of a load's rows; columns: one to sixteen a block, blocks of 8 and 9 (2,112) and of 15 and 16 (4,032);
# K: one pair of k-steps, fewer pairs than waves, one more than fills their rings, many
@pytest.mark.parametrize("m", [1, 3, 8, 9, 13, 16])
@pytest.mark.parametrize("n,k", [(256, 64), (320, 448), (1024, 2112), (2048, 512), (2112, 576), (2560, 4096), (4032, 128), (4096, 2048)])
def test_stream_and_rows(ops, m, n, k):
    residual, x = rnd(m, n, seed=1), rnd(m, k, seed=2, dtype=torch.bfloat16)
    w, weight = rnd(n, k, seed=3, scale=k ** -0.5, dtype=torch.bfloat16), 1.0 + 0.1 * rnd(n, seed=4)
    wider = rnd(208, n, seed=5, scale=n ** -0.5, dtype=torch.bfloat16)
    stream, sums, size = exact(residual, x, w, weight, wider)
    product = ops.product_for_norm(x, w)
    before, whole = residual.clone(), residual.clone()
    rows = ops.add_rmsnorm(residual, product, weight, EPS, torch.bfloat16, scaled=True)
    assert type(rows).__name__ == "ScaledRows" and tuple(rows.shape) == (m, n)
    # K additions in float32 of products that are exact there: K 2^-24 of the sum of their sizes at most
    bound = (x.double().abs() @ w.double().abs().T + before.double().abs()) * (k + 16) * 2.0 ** -24
    assert ((residual.double() - stream).abs() <= bound).all()
    got = ops.linear(rows, wider)
    # one rounding of the rows and one of the result to bfloat16 (2^-9 each), and the sums' own
    allowed = size * (2.0 ** -9 + (n + 64) * 2.0 ** -23) + sums.abs() * 2.0 ** -8
    assert ((got.double() - sums).abs() <= allowed).all()
    # whole tiles of 16 from 4,096 outputs on go to the kernel that shares the activations from 12 rows on, up to 11 rows to the few-row kernel
    for half in (88, 4096, 6160) if (n, k) == (2112, 576) else (88, 96):
        gate_up = rnd(2 * half, n, seed=half, scale=n ** -0.5, dtype=torch.bfloat16)
        _, gu, gu_size = exact(before, x, w, weight, gate_up)
        g, u = gu.split(half, 1)
        # gate and up are rounded to bfloat16 as well; silu's slope is at most 1.1, its size at most the gate's
        ge, ue = (gu_size * (2.0 ** -9 + (n + 64) * 2.0 ** -23) + gu.abs() * 2.0 ** -8).split(half, 1)
        ref = g * torch.sigmoid(g) * u
        assert ((ops.gated_linear(rows, gate_up).double() - ref).abs() <= 1.1 * ge * (u.abs() + ue) + g.abs() * ue + ref.abs() * 2.0 ** -7).all()
        limit = 0.7
        gc, uc = g.clamp(max=limit), u.clamp(-limit, limit)
        ref = gc * torch.sigmoid(1.702 * gc) * (uc + 1)
        got = ops.gated_linear(rows, gate_up, "clamped", limit)
        assert ((got.double() - ref).abs() <= 1.2 * ge * (uc.abs() + 1 + ue) + gc.abs() * ue + ref.abs() * 2.0 ** -7).all()
    # every form of the same rows: the norm's own, and what the product in planes and the norm give
    made = rows.made()
    assert ((ops.linear(made, wider).double() - sums).abs() <= allowed).all()
    plain = ops.add_rmsnorm(whole, product, weight, EPS, torch.bfloat16)
    # (in one plane the product is rounded to bfloat16)
    assert isinstance(plain, torch.Tensor) and ((whole.double() - stream).abs() <= bound + (x.double() @ w.double().T).abs() * 2.0 ** -8).all()
    # a row's bits do not depend on the rows beside it
    if m > 1:
        one = before[m - 1:].clone()
        alone = ops.add_rmsnorm(one, ops.product_for_norm(x[m - 1:].clone(), w), weight, EPS, torch.bfloat16, scaled=True)
        assert torch.equal(one, residual[m - 1:]) and torch.equal(alone.rows, rows.rows[m - 1:])


def test_what_goes_the_other_way(ops):
    """Sizes and types that the kernel does not take come as linear_for_residual gives them."""
    for m, n, k, dtype in ((17, 2560, 512, torch.bfloat16), (4, 192, 512, torch.bfloat16), (4, 4160, 512, torch.bfloat16),
                           (4, 2560, 96, torch.bfloat16), (4, 272, 512, torch.bfloat16), (4, 2560, 512, torch.float32)):
        x, w = rnd(m, k, seed=1, dtype=dtype), rnd(n, k, seed=2, dtype=dtype)
        got = ops.product_for_norm(x, w)
        assert isinstance(got, torch.Tensor) and torch.equal(got, ops.linear_for_residual(x, w)), (m, n, k, dtype)


def test_not_a_number_stays_in_its_row(ops):
    m, n, k = 5, 2560, 320
    residual, x = rnd(m, n, seed=1), rnd(m, k, seed=2, dtype=torch.bfloat16)
    w, wider = rnd(n, k, seed=3, dtype=torch.bfloat16), rnd(64, n, seed=4, dtype=torch.bfloat16)
    residual[2, 77], x[4, 5] = float("nan"), float("inf")
    rows = ops.add_rmsnorm(residual, ops.product_for_norm(x, w), rnd(n, seed=5), EPS, torch.bfloat16, scaled=True)
    out = ops.linear(rows, wider)
    assert torch.isfinite(out[[0, 1, 3]]).all() and not torch.isfinite(out[[2, 4]]).any()
