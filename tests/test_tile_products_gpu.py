"""The product of many rows by tiles through LDS, tile by tile at its edges, and the calls that come to it."""

from ctypes import c_float, c_int

import pytest
import torch

from qwen3_runtime_amd.ops.hip import BF16, F32, TILES, HipOps, OpsError, _ptr, _stream

DEV = "cuda"
STAGES = {0: 2, 1: 3, 2: 3, 3: 3, 4: 3, 5: 3, 6: 4, 7: 4, 8: 4, 9: 4, 10: 6, 11: 6, 12: 4, 13: 3}  # in flight


def rnd(*shape, seed, scale=1.0):
    g = torch.Generator().manual_seed(seed)
    return (scale * torch.randn(*shape, generator=g)).to(torch.bfloat16).to(DEV)


def close(got, want, k, rounded):
    """Sums of k products in float32: each addition errs by 2^-24 of the sum so far, at most k of them in a row, and
    a bfloat16 result by 2^-9 of itself (and of what lies nearest to a tie, so 2^-8)."""
    err = (got.double() - want).abs()
    size = want.abs().max()
    assert torch.isfinite(got).all()
    bound = k * 2.0 ** -24 * size + (2.0 ** -8 * want.abs() if rounded else 0.0)
    assert bool((err <= bound).all()), float((err - bound).max())


def launch(ops, x, w, out, tile, parts=1, act=-1, limit=0.0, row_scale=None):
    m, k = x.shape
    n = w.shape[0] // (2 if act >= 0 else 1)
    ops._check(ops.lib, ops.lib.qrt_gemm_tiles(_ptr(x), _ptr(w), _ptr(out), F32 if out.dtype == torch.float32 else BF16,
                                               c_int(m), c_int(n), c_int(k), c_int(tile), c_int(parts), c_int(act),
                                               c_float(limit), _ptr(row_scale), _stream()))


@pytest.mark.gpu
@pytest.mark.parametrize("tile", range(len(TILES)))
def test_every_tile_at_its_edges(tile):
    """One row and one past the tile, a column tile and a single MFMA tile more, bands of row tiles, and as many stages
    as fit the ring, one fewer and one more; every result in both types, in planes (some empty) and gated."""
    ops = HipOps()
    rows, columns, s = *TILES[tile][:2], STAGES[tile]
    for m, n, k in [(1, 16, 64), (rows - 1, columns, 64 * (s - 1)), (rows, columns + 16, 64 * s), (rows + 1, 2 * columns - 16, 64 * (s + 1)),
                    (17, 3 * columns, 64 * (2 * s + 1)), (2048 + rows + 5, columns + 48, 64),
                    (2100, 5776, 64 * s + 64)]:  # the last: more tiles than the compute units hold, a block makes several
        x, w = rnd(m, k, seed=1), rnd(n, k, seed=2, scale=0.05)
        want = x.double() @ w.double().T
        for dtype in (torch.bfloat16, torch.float32):
            out = torch.full((m, n), float("nan"), dtype=dtype, device=DEV)
            launch(ops, x, w, out, tile)
            close(out, want, k, dtype == torch.bfloat16)
        for parts in (2, 3, 8):
            out = torch.full((parts, m, n), float("nan"), device=DEV)
            launch(ops, x, w, out, tile, parts)
            close(out.double().sum(0), want, k, False)
        wg = rnd(2 * n, k, seed=3, scale=0.05)
        g, u = (x.double() @ wg.double().T).split(n, 1)
        gate = torch.full((m, n), float("nan"), dtype=torch.bfloat16, device=DEV)
        launch(ops, x, wg, gate, tile, act=0)
        # gate and up value are rounded to bfloat16 first (2^-8 of each), the result again; silu's slope is below 1.1
        assert bool(((gate.double() - torch.sigmoid(g) * g * u).abs() <= 2.0 ** -8 * ((1.1 * g.abs() + 2 * (torch.sigmoid(g) * g).abs()) * u.abs()) + 1e-4).all())
        scale = torch.rand(m, device=DEV)
        launch(ops, x, wg, gate, tile, act=1, limit=0.5, row_scale=scale)
        both = ops.linear(x, wg) if m <= 64 else torch.cat([x.float() @ wg.float().T]).to(torch.bfloat16)
        same = ops.gated_act(both, "clamped", 0.5, row_scale=scale).double()
        assert bool(((gate.double() - same).abs() <= 2.0 ** -5 * same.abs() + 2.0 ** -7).all())


@pytest.mark.gpu
def test_bits_depend_on_neither_rows_nor_tile():
    """Every output is one sum in the order of k: the same in every tile, beside any other rows; and a row that is not
    finite changes no other row, a weight row that is not finite no other column."""
    ops = HipOps()
    x, w = rnd(300, 640, seed=4), rnd(336, 640, seed=5, scale=0.05)
    x[7, 3], w[9, 5] = float("nan"), float("inf")
    outs = []
    for tile in range(len(TILES)):
        for rows in (300, 131):
            out = torch.empty((rows, 336), device=DEV)
            launch(ops, x[:rows], w, out, tile)
            outs.append(out)
    for out in outs:
        assert torch.equal(out[:131].nan_to_num(0.0, 1.0, -1.0), outs[0][:131].nan_to_num(0.0, 1.0, -1.0))
    bad = ~torch.isfinite(outs[0])
    assert bad[7].all() and bad[:, 9].all() and int(bad.sum()) == 336 + 300 - 1


@pytest.mark.gpu
@pytest.mark.parametrize("m", [17, 64, 65, 128, 129, 257, 700])
@pytest.mark.parametrize("n,k", [(96, 2048), (2560, 4096), (512, 64), (1040, 448)])
def test_calls_that_come_to_tiles(m, n, k):
    """linear, gated_linear and linear_for_residual with more rows than the streams of weights take, and the same with
    operands that tiles do not take (8 bytes off, K or weight rows of other sizes): the general ways, the same values."""
    ops, planes = HipOps(), HipOps(residual_planes=True)
    x, w = rnd(m, k, seed=6), rnd(2 * n, k, seed=7, scale=0.05)
    want = x.double() @ w.double().T
    assert ops._tiles_take(x, w)
    close(ops.linear(x, w), want, k, True)
    close(ops.linear(x, w, out_f32=True), want, k, False)
    for form in (ops, planes):
        got = form.linear_for_residual(x, w)
        assert got.dim() == 2 or m <= 128 or form is planes
        close(got if got.dim() == 2 else got.double().sum(0), want, k, got.dim() == 2)
        assert torch.equal(got, form.linear_for_residual(x, w))
    scale = torch.rand(m, device=DEV)
    for act, limit, rs in (("swiglu", 0.0, None), ("clamped", 0.7, None), ("swiglu", 0.0, scale)):
        got = ops.gated_linear(x, w, act, limit, row_scale=rs).double()
        same = ops.gated_act(want.to(torch.bfloat16), act, limit, row_scale=rs).double()
        # both round gate and up value to bfloat16: where sums lie at a tie, one step of 2^-8 of either
        assert bool(((got - same).abs() <= 2.0 ** -6 * same.abs() + 2.0 ** -7 * want.abs().max()).all())
    if m <= 64:  # streams of the weights, which refuse such operands
        return
    off = torch.empty(m * k + 4, dtype=torch.bfloat16, device=DEV)[4:].view(m, k)
    off.copy_(x)
    assert not ops._tiles_take(off, w)
    close(ops.linear(off, w), want, k, True)
    thin = w[: 2 * n - 8]
    assert not ops._tiles_take(x, thin)
    close(ops.linear(x, thin), want[:, : 2 * n - 8], k, True)


@pytest.mark.gpu
@pytest.mark.parametrize("first,second", [(i, j) for i in HipOps.EXPERT_TILES for j in HipOps.EXPERT_TILES
                                          if TILES[i][0] == TILES[j][0]])
@pytest.mark.parametrize("activation", ["swiglu", "relu2"])
def test_experts_by_every_tile(first, second, activation):
    """Experts with one pair past a tile, one that fills a tile, one with a single pair and one without any; widths of
    a part of a tile, over more stages than the ring holds."""
    from test_experts_gpu import close as near
    from test_experts_gpu import plain

    ops = HipOps()
    rows = TILES[first][0]
    ops.experts_tile_pairs_per_expert = 0
    ops.choose_experts_tiles = lambda *sizes: (rows, first, second)
    counts, h, inter = [rows + 1, rows, 1, 0], 448, 320
    index = torch.cat([torch.full((c, 1), e) for e, c in enumerate(counts)])
    index = index[torch.randperm(len(index), generator=torch.Generator().manual_seed(1))].int().to(DEV)
    t = index.shape[0]
    x = rnd(t, h, seed=1)
    up, down = rnd(4, (2 if activation == "swiglu" else 1) * inter, h, seed=2, scale=h ** -0.5), rnd(4, h, inter, seed=3, scale=inter ** -0.5)
    weight = torch.rand(t, 1, device=DEV)
    got = ops.moe_for_residual(x, up, down, index, weight, activation, 0.0)
    near(got, plain(x, up, down, index, weight, activation, 0.0, False).float(), 4e-3, 4e-3)


@pytest.mark.gpu
def test_what_tiles_refuse():
    ops = HipOps()
    x, w, out = rnd(70, 128, seed=1), rnd(64, 128, seed=2), torch.empty((2, 70, 64), device=DEV)
    for bad in (dict(tile=len(TILES)), dict(tile=-1), dict(tile=3, parts=0), dict(tile=3, parts=2, act=0), dict(tile=3, act=2)):
        with pytest.raises(Exception, match="gemm_tiles"):
            launch(ops, x, w, out, **bad)
    for a, b in ((x[:, :96].contiguous(), w[:, :96].contiguous()), (x, w[:40])):
        with pytest.raises(Exception, match="gemm_tiles"):
            launch(ops, a, b, out, tile=3)


@pytest.mark.gpu
@pytest.mark.parametrize("dtype", [torch.bfloat16, torch.float32])
def test_a_gated_product_refuses_an_activation_without_a_gate(dtype):
    """Its code tells the tiles of a product of another form, which would read the gate rows alone."""
    ops = HipOps()
    w = rnd(64, 128, seed=2).to(dtype)
    for m in (1, 16, 64, 300):
        with pytest.raises(OpsError, match="relu2"):
            ops.gated_linear(rnd(m, 128, seed=1).to(dtype), w, "relu2")


def test_what_the_library_keeps():
    takes = HipOps.library_takes
    assert not any(takes(m, n, k, form) for m in (65, 2048) for n in (256, 6144, 9728) for k, form in ((2560, "whole"), (9728, "planes"), (2560, "gated")))
    assert takes(2048, 6144, 4096) and not takes(1536, 6144, 4096) and not takes(2048, 10240, 5120)
    assert takes(1537, 12288, 4096, "gated") and not takes(1536, 12288, 4096, "gated")
    assert takes(4096, 12288, 2560, "gated") and takes(2500, 12288, 4096, "gated") and not takes(2500, 9728, 2560, "gated")
    assert takes(8192, 6144, 2560) and takes(2500, 4096, 12288, "planes") and takes(16384, 2560, 9728, "planes")
    assert not takes(2500, 2560, 9728, "planes") and not takes(3500, 2560, 4096, "planes")


def test_parts_of_few_rows():
    """Between the few-row kernel and the tiles of many rows, where the weight is small: a block a compute unit."""
    parts = HipOps.choose_short_parts
    assert [parts(m, 2560, 4096) for m in (16, 17, 64, 65, 128, 129)] == [0, 6, 6, 3, 3, 0]
    assert parts(48, 2560, 9728) == 6 and parts(48, 2048, 2048) == 4
    assert parts(48, 4096, 4096) == parts(48, 4096, 12288) == parts(48, 64, 64) == parts(100, 16384, 1024) == 0
    for n, k in ((16, 1024), (2560, 4096), (2064, 1600), (1040, 5888)):
        p = parts(40, n, k)
        assert p == 0 or (-(-(k // 64) // p) * (p - 1) < k // 64 and k // 64 >= 8 * p)


def test_choice_of_experts_tiles():
    """Both products' tiles have as many rows; one row tile an expert where a tile holds all that it may have."""
    for pairs, experts, hidden, inter in ((1, 16, 2560, 1536), (4082, 16, 2560, 1536), (512, 64, 2048, 768), (100_000, 8, 4096, 1024)):
        for gated in (True, False):
            rows, first, second = HipOps.choose_experts_tiles(pairs, experts, hidden, inter, gated)
            assert TILES[first][0] == TILES[second][0] == rows and {first, second} <= set(HipOps.EXPERT_TILES)
    assert HipOps.choose_experts_tiles(16 * 128, 16, 2560, 1536, True)[0] == 192


def test_choice_of_tile():
    """By the sizes alone; K is cut only for planes, in parts of eight stages and more, none of them empty."""
    assert HipOps.choose_tile(2048, 6144, 2560) == (0, 1)                     # 256 tiles of 256 x 192: one round
    assert HipOps.choose_tile(512, 9728, 2560, "gated") == (1, 1)             # 244 of 256 x 160
    tile, parts = HipOps.choose_tile(2048, 2560, 9728, "planes")
    assert TILES[tile][:2] == (256, 160) and parts == 2                       # 128 tiles in two parts
    for m in (1, 65, 129, 300, 1000, 2047, 8192, 100_000):
        for n, k in ((16, 64), (2560, 4096), (5120, 25600), (151936, 2560), (1024, 512)):
            assert HipOps.choose_tile(m, n, k)[1] == HipOps.choose_tile(m, n, k, "gated")[1] == 1
            tile, parts = HipOps.choose_tile(m, n, k, "planes")
            stages = k // 64
            each = -(-stages // parts)
            assert 0 <= tile < len(TILES) and 1 <= parts <= 8 and (parts == 1 or (each >= 8 and each * (parts - 1) < stages))


GATES = [0.0, -0.0, 1e-30, -1e-30, 1e-3, -1e-3, 1.0, -1.0, 20.0, -20.0, 51.0, -51.0, 51.25, -51.25, 87.0, -87.0, 87.5, -87.5, 88.0, -88.0,
         88.5, -88.5, -89.0, -100.0, -104.0, 1e4, -1e4, 1e30, -1e30, float("inf"), -float("inf"), float("nan")]


@pytest.mark.gpu
@pytest.mark.parametrize("act,limit", [("swiglu", 0.0), ("clamped", 0.7), ("clamped", 1e4)])
@pytest.mark.parametrize("way,up", [(way, up) for way in ("dense", "experts") for up in (2.0, -1e30, 0.0)] + [("dense", float("inf"))])
def test_gates_of_every_size(act, limit, up, way):
    """One column of K is not zero, so gate and up values are exact: small ones, those around the end of what the exponential
    and the quotient hold, infinite ones and NaN, beside ordinary ones in the same wave. Both forms of the activation
    err by a few 2^-24 before they round to bfloat16, half a step of 2^-8 each; zeros, infinities and NaN are the same. What
    stands beside them changes no result."""
    ops, n = HipOps(), 128
    gates = torch.tensor(GATES).to(torch.bfloat16)
    values = rnd(n, seed=9, scale=3.0).cpu()
    values[5: 5 + 2 * len(GATES): 2] = gates
    if way == "experts":  # the second product would carry what is not finite to every column
        bad = ~torch.isfinite(ops.gated_act(torch.cat([values, torch.full_like(values, up)])[None].to(DEV), act, limit)[0]).cpu()
        values[bad] = 1.0
    tame = torch.where(torch.isfinite(values) & (values.abs() < 50), values, torch.ones(()).to(values))

    def run(gate):
        w = torch.zeros(2 * n, 128)
        w[:n, 3], w[n:, 3] = gate, up
        w, x = w.to(torch.bfloat16).to(DEV), torch.zeros(200, 128, dtype=torch.bfloat16, device=DEV)
        x[:, 3] = 1.0
        if way == "dense":
            assert ops._tiles_take(x, w) and not ops.library_takes(200, n, 128, "gated")
            got = ops.gated_linear(x, w, act, limit)
        else:  # the second product takes each value to a column of its own
            ops.experts_tile_pairs_per_expert = 0
            one = torch.eye(n, dtype=torch.bfloat16, device=DEV)[None]
            assert ops.experts_fit(x, 128, n, w, one)
            act_of = ops.moe_for_residual(x, w[None].contiguous(), one, torch.zeros(200, 1, dtype=torch.int32, device=DEV),
                                          torch.ones(200, 1, device=DEV), act, limit)
            got = act_of[0]
        assert torch.equal(got.nan_to_num(7.0), got[:1].nan_to_num(7.0).expand_as(got))
        return got[0], ops.gated_act(w[:, 3].float().to(torch.bfloat16)[None].contiguous(), act, limit)[0]

    got, want = run(values)
    got, want = got.double(), want.double()
    assert torch.equal(torch.isnan(got), torch.isnan(want)) and torch.equal(torch.isinf(got), torch.isinf(want))
    known = torch.isfinite(want)
    assert torch.equal(got[~known].nan_to_num(7.0), want[~known].nan_to_num(7.0))
    assert torch.equal(got[known] == 0, want[known] == 0)
    assert bool(((got - want)[known].abs() <= 2.0 ** -7 * want[known].abs()).all())
    if act == "swiglu" and up == 2.0:
        g = values.to(DEV).double()
        exact = g / (1 + torch.exp(-g)) * up
        near = known & (g.abs() <= 87)
        assert bool(((got - exact)[near].abs() <= 2.0 ** -8 * exact[near].abs()).all())
    same = (tame == values).to(DEV)
    assert torch.equal(run(tame)[0].double()[same].nan_to_num(7.0), got[same].nan_to_num(7.0))


@pytest.mark.gpu
@pytest.mark.parametrize("activation", ["swiglu", "relu2"])
@pytest.mark.parametrize("given", [False, True])
def test_experts_tokens_in_several_goes(activation, given):
    """Tokens whose offsets would not fit 32 bits are taken in halves, here forced for an odd number of them: the same bits."""
    ops, (t, n, h, inter, top) = HipOps(), (77, 5, 192, 128, 3)
    ops.experts_tile_pairs_per_expert = 0
    x, weight = rnd(t, h, seed=1), torch.rand(t, top, device=DEV)
    up, down = rnd(n, (2 if activation == "swiglu" else 1) * inter, h, seed=2, scale=0.1), rnd(n, h, inter, seed=3, scale=0.1)
    index = torch.rand(t, n, generator=torch.Generator().manual_seed(4)).topk(top, -1).indices.int().to(DEV).contiguous()
    whole = ops.moe_for_residual(x, up, down, index, weight, activation, 0.0)
    ops.experts_tile_max_elements = 20 * h
    out = torch.full_like(whole, float("nan")) if given else None
    got = ops.moe_for_residual(x, up, down, index, weight, activation, 0.0, out=out)
    assert torch.equal(got, whole) and (out is None or got is out)


@pytest.mark.gpu
@pytest.mark.parametrize("first,second", [(0, 0), (16, 0), (0, 16), (16, 16)])
@pytest.mark.parametrize("activation", ["swiglu", "relu2"])
def test_experts_two_blocks_a_compute_unit(activation, first, second):
    """Both forms of the tiles of 128 x 128, in launches of more blocks than the compute units hold: an expert with one
    pair past a tile, one with a whole one, others with one or none. Sums are in the order of k, so the bits are those of every
    other tile."""
    from test_experts_gpu import close as near
    from test_experts_gpu import plain

    ops = HipOps()
    ops.experts_tile_pairs_per_expert = 0
    n, h, inter = 150, 448, 320
    counts = [129, 128, 0] + [1] * (n - 3)
    index = torch.cat([torch.full((c, 1), e) for e, c in enumerate(counts)])
    index = index[torch.randperm(len(index), generator=torch.Generator().manual_seed(1))].int().to(DEV)
    t = index.shape[0]
    x = rnd(t, h, seed=1)
    up, down = rnd(n, (2 if activation == "swiglu" else 1) * inter, h, seed=2, scale=h ** -0.5), rnd(n, h, inter, seed=3, scale=inter ** -0.5)
    weight = torch.rand(t, 1, device=DEV)
    outs = []
    for rows, tiles in ((128, (7 + first, 7 + second)), (64, (12, 12))):
        ops.choose_experts_tiles = lambda *sizes: (rows, 0, 1)  # noqa: B023
        ops.experts_product = lambda i, *sizes: (0.0, tiles[i], 1)  # noqa: B023
        outs.append(ops.moe_for_residual(x, up, down, index, weight, activation, 0.0))
    near(outs[0], plain(x, up, down, index, weight, activation, 0.0, False).float(), 4e-3, 4e-3)
    assert torch.equal(*outs)


def test_experts_of_60_to_110_pairs_take_tiles_of_128():
    """Between tiles that are mostly padding and two tiles an expert, where they give every compute unit one."""
    rows = [HipOps.choose_experts_tiles(64 * per, 64, 2048, 768, True)[0] for per in (32, 64, 80, 128)]
    assert rows == [64, 128, 128, 192] and HipOps.choose_experts_tiles(24 * 80, 24, 3072, 1280, True)[0] == 128
    assert HipOps.choose_experts_tiles(8 * 80, 8, 4096, 1024, True)[0] == 64
    assert HipOps.experts_product(7, 64 * 128, 128, 768, 2048, True)[1] == 7 + HipOps.experts_two_blocks   # 1,536 tiles: 3 rounds of 512
    assert HipOps.experts_product(7, 64 * 64, 64, 768, 2048, True)[1] == 7                                  # 768: 3 rounds of 256, not 1.5 of 512


def test_choice_of_tile_misses_none():
    """The search that leaves out what its bound excludes finds what trying everything finds."""
    import random

    def every(m, n, k, form):
        best = None
        for number, (rows, columns, resident, a, b, c) in enumerate(TILES):
            tiles = -(-m // rows) * -(-n // (columns // 2 if form == "gated" else columns))
            for parts in range(1, 9 if form == "planes" else 2):
                stages = -(-(k // 64) // parts)
                if parts > 1 and (stages < 8 or stages * (parts - 1) >= k // 64):
                    break
                load = -(-tiles * parts // 256)
                rounds = -(-load // resident)
                full = load / (resident * rounds) if 1 < load and resident > 1 else tiles * parts / (256 * resident * rounds)
                us = 3 + rounds * (c + stages * (a + b * full))
                if form == "planes":
                    us += m * n * (4 * parts if parts > 1 else 2) / 5e6
                if best is None or us < best[0]:
                    best = us, number, parts
        return best[1:]

    draw = random.Random(5)
    sizes = [(m, n, k) for m in (65, 129, 512, 2048, 8191) for n, k in ((16, 64), (2560, 9728), (6144, 2560), (5120, 25600))]
    sizes += [(draw.randint(1, 9000), 16 * draw.randint(1, 2000), 64 * draw.randint(1, 450)) for _ in range(1500)]
    for m, n, k in sizes:
        for form in ("whole", "gated", "planes"):
            assert HipOps.choose_tile(m, n, k, form) == every(m, n, k, form), (m, n, k, form)


@pytest.mark.gpu
@pytest.mark.parametrize("m", [1, 17, 48, 64])
def test_weights_used_once(m):
    """Up to 64 rows tiles of 64 x 64 load the weights as data used once, beyond as any other: the same bits."""
    ops, n, k = HipOps(), 1040, 1600
    x, w = rnd(65, k, seed=1), rnd(n, k, seed=2, scale=0.05)
    for parts in (1, 3, 8):
        outs = []
        for rows in (m, 65):
            out = torch.full((parts, rows, n) if parts > 1 else (rows, n), float("nan"), device=DEV)
            launch(ops, x[:rows], w, out, 12, parts)
            outs.append(out)
        assert torch.isfinite(outs[0]).all() and torch.equal(outs[0], outs[1][..., :m, :])
