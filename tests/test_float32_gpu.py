"""The float32 kernels at the edges of their tiles: products against float64 within the bound of a
float32 sum, equal bits however many rows share a launch; attention by tiles against the plain one."""

import copy
import math

import pytest
import torch

from plain import ops_ref as R
from test_kernels_gpu import DEV, build_attention_case, close, rnd

pytestmark = pytest.mark.gpu


@pytest.fixture(scope="module")
def ops():
    from qwen3_runtime_amd.ops.hip import HipOps

    return HipOps()


# K: less than a chunk of 16, no multiple of 16, the ends of the 4-, 8- and 16-part ranges; N and M: around 16, 64, 128
@pytest.mark.parametrize("n,k", [(1, 4), (17, 20), (64, 252), (65, 260), (130, 1028), (48, 8188), (33, 8192), (15, 10004)])
def test_product_against_float64_and_equal_bits_for_any_number_of_rows(ops, n, k):
    x, w = rnd(200, k, seed=1), rnd(n, k, seed=2, scale=0.05)
    whole = ops.linear(x, w)
    want = x.double() @ w.double().T
    # a sum of k products in any order, each rounded: at most k units of 2^-24 of the sum of magnitudes
    bound = k * 2.0 ** -24 * (x.double().abs() @ w.double().abs().T)
    assert ((whole.double() - want).abs() <= bound).all()
    for m in (1, 8, 9, 16, 17, 32, 33, 64, 65, 129):
        assert torch.equal(ops.linear(x[70: 70 + m].contiguous(), w), whole[70: 70 + m]), m


# rows: one unit of 8, its edges, the blocks of 16 and 64; weight rows: none, one and part of a block of 8; K: an end inside a slot of 32
@pytest.mark.parametrize("activation,limit", [("swiglu", 0.0), ("clamped", 0.7)])
@pytest.mark.parametrize("inter,k", [(1, 4), (12, 68), (40, 2560), (24, 8228)])
def test_gated_product_of_few_rows_has_the_bits_of_product_and_activation(ops, inter, k, activation, limit):
    x, w = rnd(33, k, seed=5), rnd(2 * inter, k, seed=6, scale=0.1)
    for m in (1, 8, 9, 16, 17, 32, 33):
        both = ops.linear(x[:m], w)
        assert torch.equal(ops.gated_linear(x[:m], w, activation, limit), ops.gated_act(both, activation, limit)), m


# weight rows: a remainder of every tile; K: groups of two and of four parts, one that K ends before, an end inside a slot of 32
@pytest.mark.parametrize("n,k", [(1, 260), (65, 1028), (2560, 264), (52, 8196)])
def test_product_in_planes_is_the_same_for_any_number_of_rows(ops, n, k):
    from qwen3_runtime_amd.ops.hip import HipOps

    planes = HipOps(residual_planes=True)
    x, w = rnd(300, k, seed=11), rnd(n, k, seed=12, scale=0.05)
    whole = planes.linear_for_residual(x, w)
    assert whole.shape == (4, 300, n)
    want = x.double() @ w.double().T
    assert ((whole.double().sum(0) - want).abs() <= k * 2.0 ** -24 * (x.double().abs() @ w.double().abs().T)).all()
    for m in (1, 8, 9, 16, 17, 32, 33, 64, 65, 129):
        assert torch.equal(planes.linear_for_residual(x[70: 70 + m].contiguous(), w), whole[:, 70: 70 + m]), m
    # the norm adds the planes' sum with one rounding
    res, weight = rnd(300, n, seed=13), torch.ones(n, device=DEV)
    total = ((whole[0] + whole[1]) + whole[2]) + whole[3]
    a, b = res.clone(), res.clone()
    assert torch.equal(ops.add_rmsnorm(a, whole, weight, 1e-6, torch.float32), ops.add_rmsnorm(b, total, weight, 1e-6, torch.float32))
    assert torch.equal(a, b)


def tile_of(m, n, groups=1):
    """The tile that the launch takes by its model of the time (in multiples of a hundredth of a round's)."""
    tiles, cost = -(-m // 128) * -(-n // 128), {}
    if groups == 1 and tiles >= 1024:
        cost[128, 128] = 0 if 64 < m <= 128 else 100 * -(-tiles // 256) * 2324   # one row of tiles
    for (tm, tn), (round_time, least) in {(64, 64): (606, 130), (64, 32): (329, 180), (32, 32): (190, 250)}.items():
        rounds = -(-(-(-m // tm) * -(-n // tn) * groups) // 256)
        cost[tm, tn] = max(100 * rounds, least) * round_time
    return min(cost, key=lambda t: (cost[t], t != (64, 64)))


# every tile that a whole product takes, a remainder of its rows and columns; K: parts of two, five and seventeen stages of 32, an odd
# number of stages in all, an end inside a stage and inside a group of four
@pytest.mark.parametrize("n,tile", [(131, (32, 32)), (2561, (64, 32)), (6148, (64, 64))])
@pytest.mark.parametrize("k", [260, 1028, 8196])
def test_whole_product_by_every_tile_has_the_bits_of_few_rows(ops, n, tile, k):
    assert tile_of(301, n) == tile
    x, w = rnd(301, k, seed=21), rnd(n, k, seed=22, scale=0.05)
    whole = ops.linear(x, w)
    bound = k * 2.0 ** -24 * (x.double().abs() @ w.double().abs().T)   # as above
    assert ((whole.double() - x.double() @ w.double().T).abs() <= bound).all()
    for first, m in ((0, 1), (60, 9), (127, 32), (269, 32)):
        assert torch.equal(ops.linear(x[first: first + m].contiguous(), w), whole[first: first + m]), (first, m)


def test_product_of_many_rows_in_large_tiles(ops):
    x, w = rnd(4100, 36, seed=3), rnd(4097, 36, seed=4)   # 65 x 65 tiles of 64, the last of four rows and one column
    whole = ops.linear(x, w)
    bound = 36 * 2.0 ** -24 * (x.double().abs() @ w.double().abs().T)
    assert ((whole.double() - x.double() @ w.double().T).abs() <= bound).all()
    assert torch.equal(ops.linear(x[4099:].contiguous(), w), whole[4099:])


# the last tile of one row and 102 columns, or of two columns; K: one stage a part, two with an odd number in all, 17
@pytest.mark.parametrize("m,n,k", [(3969, 4070, 36), (4096, 3970, 260), (4000, 4066, 8196), (100, 131100, 36)])
def test_product_of_many_rows_in_tiles_of_128(ops, m, n, k):
    assert tile_of(m, n) == (128, 128)
    x, w = rnd(m, k, seed=3), rnd(n, k, seed=4, scale=0.05)
    whole = ops.linear(x, w)
    for first in (0, m // 3, m - 32):
        part = x[first: first + 32].contiguous()
        assert torch.equal(ops.linear(part, w), whole[first: first + 32]), first
        bound = k * 2.0 ** -24 * (part.double().abs() @ w.double().abs().T)   # as above
        assert ((whole[first: first + 32].double() - part.double() @ w.double().T).abs() <= bound).all()


# 64 x 64 and 128 x 128, remainders of rows and columns; K: groups of two parts of two stages, the third of one part and the fourth of none;
# of two parts of five; of four of seventeen
@pytest.mark.parametrize("m,n,k", [(2049, 2563, 260), (1281, 5123, 1028), (3969, 4070, 1028), (4090, 4096, 8196)])
def test_product_for_the_residual_of_many_rows_or_few_of_a_tall_weight_comes_added_up(ops, m, n, k):
    """One matrix in place of four planes, with the bits of the planes' sum, so that a row's stream and norm do not go by the number of rows."""
    from qwen3_runtime_amd.ops.hip import HipOps

    planes = HipOps(residual_planes=True)
    x, w = rnd(m, k, seed=11), rnd(n, k, seed=12, scale=0.05)
    whole = planes.linear_for_residual(x, w)
    assert whole.shape == (m, n)
    res, weight = rnd(m, n, seed=13), torch.ones(n, device=DEV)
    stream = res.clone()
    normed = ops.add_rmsnorm(stream, whole, weight, 1e-6, torch.float32)
    for first, rows in ((0, 1), (63, 9), (300, 17), (400, 32), (130, 33), (m - 200, 200)):
        at = slice(first, first + rows)
        few = planes.linear_for_residual(x[at].contiguous(), w)
        assert few.shape == ((rows, n) if n >= 4096 and rows <= 32 else (4, rows, n))   # few rows: by the weight's
        assert torch.equal(few if few.dim() == 2 else ((few[0] + few[1]) + few[2]) + few[3], whole[at]), (first, rows)
        part = res[at].clone()
        assert torch.equal(ops.add_rmsnorm(part, few, weight, 1e-6, torch.float32), normed[at])
        assert torch.equal(part, stream[at])
        bound = k * 2.0 ** -24 * (x[at].double().abs() @ w.double().abs().T)   # as above
        assert ((whole[at].double() - x[at].double() @ w.double().T).abs() <= bound).all()


@pytest.mark.parametrize("k,planes", [(4, False), (256, True)])
def test_product_of_more_rows_than_a_grid_has_tiles(k, planes):
    """65,535 rows of tiles of 64 are 4,194,240; the tiles beyond are in a launch of their own."""
    from qwen3_runtime_amd.ops.hip import HipOps

    ops, m, n = HipOps(residual_planes=planes), 65535 * 64 + 70, 3
    gen = torch.Generator(DEV).manual_seed(1)
    x, w = torch.randn(m, k, device=DEV, generator=gen), rnd(n, k, seed=2)
    product = ops.linear_for_residual if planes else ops.linear
    got = product(x, w)
    assert got.shape == (m, n)
    for first in (0, 65535 * 64 - 40, 65535 * 64 - 1, m - 64):
        few = product(x[first: first + 64].contiguous(), w)
        few = ((few[0] + few[1]) + few[2]) + few[3] if planes else few
        assert torch.equal(few, got[first: first + 64]), first
    close(got, x @ w.T, 1e-5 * math.sqrt(k), 1e-5)


@pytest.mark.parametrize("seqs,nq,nkv,d,dv,ps,more", [
    ([(1, 16), (1, 17), (1, 130)], 4, 2, 128, 128, 16, {}),                       # decoding: eight waves share the keys
    ([(20, 33), (7, 7), (1, 1)], 5, 1, 48, 48, 4, {}),                            # a tile's 16 rows cut a token's heads
    ([(300, 300), (160, 190)], 8, 8, 32, 16, 24, {}),                             # many tiles: four waves; values of another size
    ([(40, 90)], 4, 2, 256, 256, 8, {"window": 9, "keep_first": 5, "sink": True}),
    ([(1, 99), (33, 99)], 6, 2, 64, 80, 16, {"window": 40, "softcap": 5.0}),
    ([(50, 75)], 4, 4, 16, 32, 12, {"chunk": 24, "gate": True}),
])
def test_attention_by_tiles(ops, seqs, nq, nkv, d, dv, ps, more):
    more = dict(more)
    q, cache, ctx = build_attention_case(seqs, nq, nkv, d, ps, torch.float32, window=more.get("window"), poison=True)
    if dv != d:
        cache.v = rnd(cache.v.shape[0], nkv, dv, ps, seed=7)
    if more.pop("gate", False):
        more["gate"] = rnd(ctx.num_tokens, nq * dv, seed=9)
    window, scale = more.pop("window", None), 1.0 / math.sqrt(d)
    want = R.paged_attention(q.double(), cache.k, cache.v, ctx.cu_q.cpu(), ctx.kv_lens.cpu(), cache.group.block_table, ps,
                             nq, nkv, d, scale, window, torch.float64, value_dim=dv, **more)
    got = ops.paged_attention(q, cache, ctx, nq, nkv, d, scale, window, value_dim=dv, **more)
    # scores of size 3 * sqrt(d) * scale and values of size 3: sums of up to 300 float32 terms
    close(got, want.float(), 2e-5, 2e-5)


@pytest.mark.parametrize("value", [float("inf"), float("-inf"), float("nan")])
@pytest.mark.parametrize("nq,nkv,d,more", [(4, 2, 128, {}), (8, 8, 32, {"window": 23}), (6, 1, 256, {"window": 40, "keep_first": 5}), (4, 4, 64, {"chunk": 32})])
def test_attention_takes_nothing_from_keys_a_token_does_not_see(ops, value, nq, nkv, d, more):
    """A value and a key of one token that are not finite: tokens that do not see it are as they are without it (but for the
    order of their sums)."""
    n = 75
    q, cache, ctx = build_attention_case([(n, n), (1, n)], nq, nkv, d, 16, torch.float32)
    attend = lambda cache: ops.paged_attention(q, cache, ctx, nq, nkv, d, d ** -0.5, more.get("window"), chunk=more.get("chunk"),  # noqa: E731
                                               keep_first=more.get("keep_first", 0))
    want, pos = attend(cache), torch.arange(n, device=DEV)
    for at in (0, 3, 16, 37, 74):
        sees = pos >= at
        if "window" in more:
            sees &= (pos - at < more["window"]) | (at < more.get("keep_first", 0))
        if "chunk" in more:
            sees &= pos // 32 == at // 32
        for stream in ("v", "k"):
            odd = copy.copy(cache)
            odd.k, odd.v = k, v = cache.k.clone(), cache.v.clone()
            for s in (0, 1):
                page, off = int(cache.group.block_table[s, at // 16]), at % 16
                if stream == "v":
                    v[page, :, d - 1, off] = value
                else:
                    k[page, :, off, 0] = value
            got = attend(odd)
            close(got[:n][~sees], want[:n][~sees], 2e-5, 2e-5)
            if not bool(sees[n - 1]):
                close(got[n], want[n], 2e-5, 2e-5)


def test_a_first_key_of_no_weight_leaves_a_token_its_other_keys(ops):
    """Token 16 alone sees key 16, whose score is minus infinity for all heads: its other sixteen keys count as ever."""
    q, cache, ctx = build_attention_case([(17, 17)], 2, 2, 32, 16, torch.float32)
    q.view(17, 2, 32)[16] = q.view(17, 2, 32)[16].abs()
    page = int(cache.group.block_table[0, 1])
    cache.k[page, :, 0, :] = float("-inf")
    got = ops.paged_attention(q, cache, ctx, 2, 2, 32, 0.2, None).view(17, 2, 32)[16]
    page = int(cache.group.block_table[0, 0])
    k, v = cache.k[page].cpu().double(), cache.v[page].cpu().double()
    p = torch.softmax((q.view(17, 2, 32)[16].cpu().double()[:, None, :] * k).sum(-1) * 0.2, -1)
    close(got, (p[:, None, :] * v).sum(-1).float(), 2e-5, 2e-5)


@pytest.mark.parametrize("nq,nkv,d,window,keep", [(4, 2, 128, 40, 0), (6, 1, 64, 33, 0), (2, 2, 256, 50, 21), (8, 8, 16, 17, 5)])
def test_attention_where_pages_in_front_of_the_window_were_given_back(ops, nq, nkv, d, window, keep):
    seqs = [(1, 200), (30, 150), (70, 300), (5, 20)]
    q, cache, ctx = build_attention_case(seqs, nq, nkv, d, 16, torch.float32, window=window, poison=True)
    attend = lambda: ops.paged_attention(q, cache, ctx, nq, nkv, d, d ** -0.5, window, keep_first=keep)  # noqa: E731
    want = R.paged_attention(q.double(), cache.k, cache.v, ctx.cu_q.cpu(), ctx.kv_lens.cpu(), cache.group.block_table, 16,
                             nq, nkv, d, d ** -0.5, window, torch.float64, keep_first=keep)
    table = cache.group.block_table.clone()
    for s, (n, kv) in enumerate(seqs):
        for p in range(-(-keep // 16), max(0, kv - n - window + 1) // 16):
            cache.k[int(table[s, p])] = cache.v[int(table[s, p])] = float("nan")   # its next holder's
            table[s, p] = -1
    cache.group.block_table = table
    close(attend(), want.float(), 2e-5, 2e-5)
