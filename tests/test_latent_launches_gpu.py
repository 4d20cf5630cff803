"""Steps of latent attention and retention that share a launch (csrc/latent.hip), against the same steps one by one: the same bits."""

import pytest
import torch

pytestmark = pytest.mark.gpu
DEV = "cuda:0"


@pytest.fixture(scope="module")
def ops():
    from qwen3_runtime_amd.ops.hip import HipOps

    return HipOps()


def rnd(*shape, seed, dtype=torch.bfloat16):
    return torch.randn(*shape, generator=torch.Generator().manual_seed(seed)).to(dtype).to(DEV)


def positions(t):
    return (torch.arange(t, dtype=torch.int32) * 37 % 5000).to(DEV)


# one and eight tokens, a tile and one more, rows that come in rounds of 512 tokens; outputs of one narrow tile, of one and a part
@pytest.mark.parametrize("t", [1, 8, 129, 513])
@pytest.mark.parametrize("heads,k,n,rot", [(3, 64, 48, 16), (32, 128, 384, 64), (2, 192, 132, 8), (2, 64, 20, 12)])
def test_products_per_head_with_a_gate_and_beside_a_rotation(ops, t, heads, k, n, rot):
    x, w = rnd(t, heads * (k + rot), seed=1), rnd(heads, n, k, seed=2)
    freq = (10000.0 ** (-torch.arange(rot // 4, dtype=torch.float32) / 8)).to(DEV)
    width = n + rot
    apart, together = torch.zeros(t, heads * width, dtype=torch.bfloat16, device=DEV), torch.zeros(t, heads * width, dtype=torch.bfloat16, device=DEV)
    for extra in ({}, {"neighbours": True, "magnitude": 1.25}):
        rotation = dict(in_stride=k + rot, in_offset=k, out_stride=width, out_offset=n, heads=heads, width=rot, positions=positions(t), freq=freq, **extra)
        ops.heads_linear(x, k + rot, 0, w, apart, width, 0)
        ops.rotate_half(x, out=apart, **rotation)
        ops.heads_linear(x, k + rot, 0, w, together, width, 0, rotation=rotation)
        assert torch.equal(apart, together)
    gates = rnd(t, 5 + heads * n + 7, seed=3)
    for first in (0, 4, 5):  # a column that is no whole piece of eight bytes goes through the pass of its own
        gate = gates[:, first: first + heads * n]
        want, got = (torch.empty(t, heads * n, dtype=torch.bfloat16, device=DEV) for _ in range(2))
        ops.sigmoid_gate(ops.heads_linear(x, k + rot, 0, w, want, n, 0), gate)
        ops.heads_linear(x, k + rot, 0, w, got, n, 0, gate=gate)
        assert torch.equal(want, got)


@pytest.mark.parametrize("dtype", [torch.bfloat16, torch.float32])
@pytest.mark.parametrize("t,q_rank,rank,rot", [(1, 768, 384, 64), (9, 1030, 1500, 6), (40, 24, 8, 0)])
def test_the_cached_row_and_a_norm(ops, dtype, t, q_rank, rank, rot):
    from qwen3_runtime_amd.parts.base import CacheView, GroupView
    from qwen3_runtime_amd.parts.plan import CacheSpec

    y, ps, pages = rnd(t, q_rank + rank + rot + 3, seed=1, dtype=dtype), 16, 8
    wq, w = rnd(q_rank, seed=2, dtype=torch.float32), rnd(rank, seed=3, dtype=torch.float32)
    freq = (100.0 ** (-torch.arange(rot // 2, dtype=torch.float32) / 8)).to(DEV) if rot else None
    slots = torch.randperm(ps * pages, generator=torch.Generator().manual_seed(4))[:t].to(torch.int32).to(DEV)
    caches = []
    for norm in (None, (0, q_rank, wq)):
        k = torch.zeros(pages, 1, ps, rank + rot, dtype=dtype, device=DEV)
        v = torch.zeros(pages, 1, rank + rot, ps, dtype=dtype, device=DEV)
        view = CacheView(CacheSpec("paged_kv", heads=1, head_dim=rank + rot), True, GroupView(ps, None, None, slots), k, v)
        got = ops.latent_store(y, q_rank, rank, rot, w, 1e-5, positions(t), freq, view, norm=norm)
        caches.append((k, v))
    assert torch.equal(caches[0][0], caches[1][0]) and torch.equal(caches[0][1], caches[1][1])
    assert torch.equal(got, ops.rmsnorm_columns(y, 0, q_rank, wq, 1e-5))
    x = y[:, :q_rank].double()
    want = x / torch.sqrt(x.square().mean(-1, keepdim=True) + 1e-5) * wq.double()
    assert ((got.double() - want).abs() <= want.abs() * (2.0 ** -8 if dtype == torch.bfloat16 else (q_rank + 16) * 2.0 ** -24)).all()


# heads in whole pieces of eight elements and others; eight tokens and more of them
@pytest.mark.parametrize("t,heads,dim,vdim,pairs", [(1, 4, 64, 128, 32), (8, 32, 128, 128, 64), (9, 3, 40, 24, 16), (5, 3, 20, 12, 10), (600, 2, 64, 64, 8)])
@pytest.mark.parametrize("dtype", [torch.bfloat16, torch.float32])
def test_queries_keys_and_values_for_retention(ops, t, heads, dim, vdim, pairs, dtype):
    y = rnd(t, 2 * heads * dim + heads * vdim + 8, seed=1, dtype=dtype)
    freq = (1000.0 ** (-torch.arange(pairs, dtype=torch.float32) / pairs)).to(DEV)
    got = ops.retention_prepare(y, heads, dim, vdim, positions(t), freq, dim ** -0.5)
    want = torch.empty_like(got)
    ops.rotate_half(y, dim, 0, want, dim, 0, 2 * heads, dim, positions(t), freq, scale_from_head=heads, scale=dim ** -0.5)
    want[:, 2 * heads * dim:] = y[:, 2 * heads * dim: 2 * heads * dim + heads * vdim].float()
    # sines of the two rotations are of the same angles, but a product and a sum may be joined in one kernel and not in the other
    assert ((got - want).abs() <= 4e-7 * want.abs().max()).all()
