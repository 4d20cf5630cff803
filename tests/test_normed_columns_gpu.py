"""The norm of some columns at the edges of the pieces that a row is read in (csrc/latent.hip), against float64."""

import pytest
import torch

from test_kernels_gpu import rnd

pytestmark = pytest.mark.gpu


@pytest.fixture(scope="module")
def ops():
    from qwen3_runtime_amd.ops.hip import HipOps

    return HipOps()


# pieces of 256 elements: one to four stay in registers, four at a time come again beyond, and one to four at the end
@pytest.mark.parametrize("dtype", [torch.float32, torch.bfloat16])
@pytest.mark.parametrize("width", [1, 255, 256, 257, 512, 513, 768, 769, 1024, 1025, 1280, 1537, 2048, 2049, 2050, 3300])
def test_normed_columns(ops, dtype, width):
    y, weight = rnd(3, width + 7, seed=1, dtype=dtype), 1.0 + 0.1 * rnd(width, seed=2)
    y[1] *= 1e-3
    got = ops.rmsnorm_columns(y, 5, width, weight, 1e-6)
    x = y[:, 5: 5 + width].double()
    want = x / (x.square().mean(-1, keepdim=True) + 1e-6).sqrt() * weight.double()
    # the sum's relative error is at most (adds a thread + adds over the block) 2^-24, of which the root takes half; five more roundings, and the result's:
    # bfloat16 has 8 bits, so half a unit of the last is up to 2^-8 of the value
    bound = (width / 512 + 16 + 6) * 2.0 ** -24 + (2.0 ** -8 if dtype == torch.bfloat16 else 0.0)
    assert ((got.double() - want).abs() <= want.abs() * bound).all()
