"""The router's choice at the edges of the pieces that a row is asked for in (csrc/moe.hip)."""

import pytest
import torch

from test_kernels_gpu import DEV, rnd

pytestmark = pytest.mark.gpu


@pytest.fixture(scope="module")
def ops():
    from qwen3_runtime_amd.ops.hip import HipOps

    return HipOps()


# pieces of 256: part of one, one, one and a bit, four, five, twelve (all at one time up to 256 tokens), thirteen in two rounds, 25 in three
@pytest.mark.parametrize("dtype", [torch.float32, torch.bfloat16])
@pytest.mark.parametrize("tokens", [1, 256, 257])
@pytest.mark.parametrize("hidden", [4, 252, 256, 260, 1024, 1028, 3072, 3076, 6148])
def test_scores_of_every_expert(ops, dtype, tokens, hidden):
    x, router = rnd(tokens, hidden, seed=1, dtype=dtype), rnd(17, hidden, seed=2, scale=hidden ** -0.5)
    index, weight = ops.route_top(x, router, None, 17, scoring="sigmoid")
    logits, size = x.double() @ router.double().T, x.double().abs() @ router.double().abs().T
    assert torch.equal(index.sort(dim=1).values, torch.arange(17, device=DEV, dtype=torch.int32).expand(tokens, 17))
    want, off = (v.gather(1, index.long()) for v in (logits.sigmoid(), size))
    # a sum of `hidden` products in float32, a quarter of its error as the sigmoid's slope is at most that, and the sigmoid's own
    assert ((weight.double() - want).abs() <= off * hidden * 2.0 ** -26 + 2.0 ** -22).all()
    assert (weight[:, 1:] <= weight[:, :-1]).all()
