"""Products per head by tiles (csrc/latent.hip) on both sides of where the tiles of few tokens begin, against float64."""

import pytest
import torch

pytestmark = pytest.mark.gpu
DEV = "cuda:0"


# tiles of 32 tokens by 64 outputs: one, some, 256, and a token or an output more; K of one stage, of the ring's eight, of one more and of several rings
@pytest.mark.parametrize("heads,n,t", [(1, 20, 1), (3, 132, 33), (32, 128, 128), (32, 128, 129), (128, 128, 32), (16, 1024, 32), (16, 1028, 31)])
@pytest.mark.parametrize("k", [64, 448, 512, 576, 1344])
def test_every_product(heads, n, t, k):
    from qwen3_runtime_amd.ops.hip import HipOps

    ops, g = HipOps(), torch.Generator().manual_seed(heads * 7 + k)
    x = torch.randn(t, heads * (k + 8), generator=g).to(torch.bfloat16).to(DEV)
    w = (torch.randn(heads, n, k, generator=g) * k ** -0.5).to(torch.bfloat16).to(DEV)
    gate = torch.randn(t, heads * n, generator=g).to(torch.bfloat16).to(DEV)
    out, gated = (torch.full((t, heads * n), float("nan"), dtype=torch.bfloat16, device=DEV) for _ in range(2))
    ops.heads_linear(x, k + 8, 8, w, out, n, 0)
    ops.heads_linear(x, k + 8, 8, w, gated, n, 0, gate=gate)
    xs = x.double().view(t, heads, k + 8)[:, :, 8:].transpose(0, 1).contiguous()
    wt = w.double().transpose(1, 2).contiguous()
    want, size = torch.bmm(xs, wt).transpose(0, 1), torch.bmm(xs.abs(), wt.abs()).transpose(0, 1)
    # K additions in float32 of products that are exact there, and the result's rounding to bfloat16
    assert ((out.double().view(t, heads, n) - want).abs() <= size * (k + 16) * 2.0 ** -24 + want.abs() * 2.0 ** -8).all()
    assert torch.equal(gated, ops.sigmoid_gate(out, gate))
