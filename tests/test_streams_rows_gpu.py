"""The step between two sub-layers over several residual streams: every number of planes and of streams that the
kernel knows when compiling, and the rows around its widths."""

from types import SimpleNamespace

import pytest
import torch

from qwen3_runtime_amd.ops.hip import HipOps

pytestmark = pytest.mark.gpu
DEV = "cuda"


def rnd(*shape, seed, scale=1.0):
    return (scale * torch.randn(*shape, generator=torch.Generator().manual_seed(seed))).to(DEV)


@pytest.mark.parametrize("t,h,s", [(1, 64, 4), (3, 260, 5), (600, 2560, 4), (2, 4096, 8), (5, 4100, 4), (2, 8192, 3), (4, 1001, 2),
                                   (2, 4099, 8)])
@pytest.mark.parametrize("planes", [0, 1, 2, 3, 4, 5, 6, 7, 8, 9])
def test_mix_norm(t, h, s, planes):
    ops = HipOps()
    x = rnd(t, s, h, seed=1)
    w, b, read = rnd(h, seed=2), rnd(h, seed=3), rnd(s, seed=4)
    mix, out, y = (0.5 * rnd(s, s, seed=5), rnd(s, seed=6), rnd(planes, t, h, seed=7)) if planes else (None, None, None)
    new = x.double()
    if planes:
        new = torch.einsum("st,nsh->nth", mix.double(), new) + out.double()[:, None] * y.double().sum(0)[:, None, :]
    u = torch.einsum("t,nth->nh", read.double(), new)
    u = u - u.mean(-1, keepdim=True)
    want = u / torch.sqrt(u.square().mean(-1, keepdim=True) + 1e-6) * w.double() + b.double()
    got_x = x.clone()
    update = SimpleNamespace(y=y[0] if planes == 1 else y, mix=mix, out=out) if planes else None
    got = ops.mix_norm(got_x, update, read, w, b, 1e-6, torch.float32)
    # float32 sums of at most 8 + 9 + 8 terms of size one to four for a stream, of h of them for a row's mean and variance
    assert (got_x.double() - new).abs().max() <= 32 * 2.0 ** -24 * new.abs().max()
    assert (got.double() - want).abs().max() <= (64 + h ** 0.5) * 2.0 ** -24 * max(1.0, float(want.abs().max())) * 4
    # a token's values are the same whatever is beside it
    if t > 1:
        one = x[:1].clone()
        part = SimpleNamespace(y=(y[0] if planes == 1 else y)[..., :1, :].contiguous(), mix=mix, out=out) if planes else None
        assert torch.equal(ops.mix_norm(one, part, read, w, b, 1e-6, torch.float32), got[:1]) and torch.equal(one, got_x[:1])
