"""What the engine does with products of many rows for the residual: float32 planes of tiles cut along K, in every kernel
that adds planes, against float64."""

from types import SimpleNamespace

import pytest
import torch

from qwen3_runtime_amd.ops.hip import HipOps

pytestmark = pytest.mark.gpu
DEV = "cuda"
EPS = 1e-6


def rnd(*shape, seed, scale=1.0, dtype=torch.float32):
    return (scale * torch.randn(*shape, generator=torch.Generator().manual_seed(seed))).to(dtype).to(DEV)


def rms(x, w, groups=1):
    parts = x.view(x.shape[0], groups, -1)
    return (parts / torch.sqrt(parts.square().mean(-1, keepdim=True) + EPS)).view_as(x) * w.double()


@pytest.fixture(scope="module", params=[(40, 2560, 4096), (129, 2560, 4096), (200, 1040, 2048), (333, 2560, 9728), (600, 2048, 2048), (600, 5120, 5120)],
                ids=lambda p: f"{p[0]}x{p[1]}x{p[2]}")
def product(request):
    """The engine's own route: the planes, and the float64 product they add up to."""
    m, n, k = request.param
    x, w = rnd(m, k, seed=1, dtype=torch.bfloat16), rnd(n, k, seed=2, scale=k ** -0.5, dtype=torch.bfloat16)
    ops = HipOps(residual_planes=True)
    y = ops.linear_for_residual(x, w)
    assert y.dim() == 3 and 1 < y.shape[0] <= 8 and y.dtype == torch.float32
    return ops, y, x.double() @ w.double().T, 2.0 ** -24 * k


def near(got, want, bound, last=0.0):
    """``bound``: what the float32 sums may be off, in units of one; ``last``: of the result's own size, where it is rounded."""
    err = (got.double() - want).abs()
    assert torch.isfinite(got).all() and bool((err <= bound * want.abs().clamp(min=1.0) + last * want.abs()).all()), float((err - bound).max())


@pytest.mark.parametrize("some", [False, True])
def test_add_and_norms(product, some):
    """Residual add and norm, plain and behind a norm of the sub-layer's own, over all rows and over some. Sums of k products
    err by 2^-24 each; a norm divides by an rms near one, so that its results err by a few times as much."""
    ops, y, want, off = product
    m, n = want.shape
    residual, w, after = rnd(m, n, seed=3), 1 + 0.1 * rnd(n, seed=4), 1 + 0.1 * rnd(n, seed=5)
    rows = torch.tensor([m - 1, 0, m // 2], dtype=torch.int32, device=DEV) if some else None
    of = slice(None) if rows is None else rows.long()
    for scale, first in ((0.7, None), (1.0, (after, EPS))):
        sums = residual.double() + (scale * want if first is None else rms(want, after))
        got_r = residual.clone()
        got = ops.add_rmsnorm(got_r, y, w, EPS, torch.float32, rows=rows, delta_scale=scale, delta_norm=first)
        near(got, rms(sums, w)[of], 8 * off)
        near(got_r, residual.double() if some else sums, 4 * off)
        half = ops.add_rmsnorm(residual.clone(), y, w, EPS, torch.bfloat16, rows=rows, delta_scale=scale, delta_norm=first)
        near(half, rms(sums, w)[of], 8 * off, 2.0 ** -8)


def test_scaled_outputs_and_groups(product):
    ops, y, want, off = product
    m, n = want.shape
    residual, w, one, two, vector = rnd(m, n, seed=3), 1 + 0.1 * rnd(n, seed=4), rnd(n, seed=5), rnd(n, seed=6), rnd(n, seed=7)
    other = rnd(m, n, seed=8, dtype=torch.bfloat16)
    sums = residual.double() + want * one.double() + other.double() * two.double() + vector.double()
    got_r = residual.clone()
    got = ops.scaled_add_rmsnorm(got_r, [(y, one), (other, two)], w, EPS, torch.float32, vector=vector)
    near(got_r, sums, 8 * off)
    near(got, rms(sums, w), 16 * off)
    for groups in (1, 4):
        for after, norm in ((None, (w, EPS)), ((w, EPS), (w, EPS)), ((w, EPS), None)):
            add = want if after is None else rms(want, w, groups)
            got_r = residual.clone()
            got = ops.group_norm_update(got_r, y, after, norm, groups, torch.float32)
            near(got_r, residual.double() + add, 8 * off)
            near(got, residual.double() + add if norm is None else rms(residual.double() + add, w, groups), 16 * off)


@pytest.mark.parametrize("streams", [2, 4])
def test_several_residual_streams(product, streams):
    ops, y, want, off = product
    m, n = want.shape
    x, w, b = rnd(m, streams, n, seed=3), 1 + 0.1 * rnd(n, seed=4), rnd(n, seed=5)
    mix, out, read = torch.eye(streams, device=DEV) + 0.1 * rnd(streams, streams, seed=6), rnd(streams, seed=7), 1 + 0.1 * rnd(streams, seed=8)
    new = torch.einsum("st,nsh->nth", mix.double(), x.double()) + out.double()[:, None] * want[:, None]
    u = torch.einsum("t,nth->nh", read.double(), new)
    got_x = x.clone()
    got = ops.mix_norm(got_x, SimpleNamespace(y=y, mix=mix, out=out), read, w, None, EPS, torch.float32)
    near(got_x, new, 16 * off)
    near(got, rms(u, w), 32 * off)
    d = u - u.mean(-1, keepdim=True)
    near(ops.mix_norm(x.clone(), SimpleNamespace(y=y, mix=mix, out=out), read, w, b, EPS, torch.float32), rms(d, w) + b.double(), 32 * off)


def test_sums_and_means(product):
    ops, y, want, off = product
    m, n = want.shape
    acc, residual, wa, wb = rnd(m, n, seed=3), rnd(m, n, seed=4), 1 + 0.1 * rnd(n, seed=5), 1 + 0.1 * rnd(n, seed=6)
    other = rnd(m, n, seed=7, dtype=torch.bfloat16)
    near(ops.accumulate(acc.clone(), y), acc.double() + want, 4 * off)
    near(ops.norm_mean(y, wa, other, wb, EPS), 0.5 * (rms(want, wa) + rms(other.double(), wb)), 8 * off)
    near(ops.norm_mean(other, wa, y, wb, EPS), 0.5 * (rms(other.double(), wa) + rms(want, wb)), 8 * off)
    near(ops.add_concat(residual, y, 0.5, acc, torch.float32), torch.cat([residual.double() + 0.5 * want, acc.double()], 1), 4 * off)


@pytest.mark.parametrize("n,k", [(2560, 4096), (4096, 4096), (2048, 1024), (2560, 512)])
def test_the_route_of_the_engine(n, k):
    """By rows: the few-row kernel, short tiles or the kernel that shares the activations, tiles; the library beyond 2,048
    rows where it fills its own."""
    ops, w = HipOps(residual_planes=True), rnd(n, k, seed=2, scale=k ** -0.5, dtype=torch.bfloat16)
    for m in (1, 8, 9, 16, 17, 64, 65, 128, 129, 700, 2048, 2049):
        x = rnd(m, k, seed=m, dtype=torch.bfloat16)
        kernel, short = ops._own_kernel(m, n, k, "planes"), ops.choose_short_parts(m, n, k)
        if kernel is None:
            parts = 1 if ops.library_takes(m, n, k, "planes") else ops.choose_tile(m, n, k, "planes")[1]
        else:
            parts = short or ops.choose_k_parts(n, k, m, kernel == 1)
        y = ops.linear_for_residual(x, w)
        assert (y.shape[0] if y.dim() == 3 else 1) == parts and (y.dim() == 3) == (parts > 1)
        want = x.double() @ w.double().T
        near(y.sum(0) if parts > 1 else y, want, 2.0 ** -24 * k, 0.0 if parts > 1 else 2.0 ** -8)


@pytest.mark.parametrize("name", ["qwen3_4b", "deginex_4b_moe", "roserax_2b", "zisedra_2b", "zuvasun_2b", "sarudra_2b", "dekinex_2b"])
def test_whole_models_with_and_without(name):
    """A few layers of every design at the sizes it is run at, a prompt of 333 tokens and portions behind it: with the engine's ops
    and with those that hand products of many rows over as one bfloat16 matrix, both beside the same engine in float32. Planes round
    less, so their error is no larger but for chance (a rounding that moves a token to another expert moves its logits in
    either): the middle token's by a quarter. A plane lost or added twice would move every token by a sizeable part of its logits."""
    from qwen3_runtime_amd.engine.batch import StepEntry
    from qwen3_runtime_amd.llm import build_engine
    from qwen3_runtime_amd.registry import preset_config

    raw = dict(preset_config(name))
    if isinstance(raw.get("layers"), list):
        raw["layers"] = raw["layers"][:4]
    else:
        raw["num_hidden_layers"] = 3
    ids = torch.randint(0, 2000, (500,), generator=torch.Generator().manual_seed(2)).tolist()

    def logits(engine):
        engine.cache.admit("a")
        rows = [engine.runner.step([StepEntry("a", ids[p:q], list(range(0, q - p, 7)))]) for p, q in ((0, 333), (333, 463), (463, 500))]
        engine.cache.release("a")
        return torch.cat([r.float() if isinstance(r, torch.Tensor) else torch.stack(list(r.values())).float() for r in rows])

    got = {}
    for dtype in ("float32", "bfloat16"):
        engine = build_engine(None, config=raw, seed=5, dtype=dtype, block_size=16, num_kv_blocks=80, max_num_seqs=2,
                              max_num_batched_tokens=512, max_model_len=1024, cuda_graph=False)
        ops, made = engine.runner.ops, []
        assert ops.residual_planes
        inner = ops.linear_for_residual
        ops.linear_for_residual = lambda x, w: (made.append(inner(x, w)), made[-1])[1]  # noqa: B023
        for planes in (True, False) if dtype == "bfloat16" else (None,):
            ops.residual_planes = bool(planes)
            made.clear()
            got[planes] = logits(engine)
            assert (3 in [y.dim() for y in made if y.shape[-2] > 128]) == bool(planes)
    want = got.pop(None)
    err = {planes: float(((rows - want).square().mean(-1).sqrt() / want.std(-1)).median()) for planes, rows in got.items()}
    print(name, err)
    assert torch.isfinite(got[True]).all() and err[True] <= 1.25 * err[False], err
