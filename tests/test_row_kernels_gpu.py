"""Row passes that load whole pieces of a row: the norm behind a sub-layer with the sum and the next norm, the
router's choice with a lane per expert, rotation by pieces, the squared relu; against the plain forms, at widths and
numbers of rows on both sides of every choice between their variants."""

import pytest
import torch

from plain import ops_ref as R
from test_kernels_gpu import DEV, close, rnd

pytestmark = pytest.mark.gpu


@pytest.fixture(scope="module")
def ops():
    from qwen3_runtime_amd.ops.hip import HipOps

    return HipOps()


@pytest.mark.parametrize("t,h", [(3, 4), (5, 1020), (511, 2048), (512, 2052), (513, 3072), (600, 3076), (7, 4096), (4, 4100), (3, 37)])
@pytest.mark.parametrize("planes,dtype", [(1, torch.bfloat16), (2, torch.float32), (5, torch.float32)])
def test_norm_add_rmsnorm(ops, t, h, planes, dtype):
    y = rnd(*((t, h) if planes == 1 else (planes, t, h)), dtype=dtype, seed=1)
    residual, after, weight = rnd(t, h, seed=2), rnd(h, seed=3), rnd(h, seed=4)
    rows = torch.tensor([t - 1, 0], dtype=torch.int32, device=DEV)
    for picked in (rows, None):
        got_r, want_r = residual.clone(), residual.double()
        got = ops.add_rmsnorm(got_r, y, weight, 1e-5, torch.float32, rows=picked, delta_norm=(after, 1e-6))
        d = y.double().sum(0) if y.dim() == 3 else y.double()
        d = d * torch.rsqrt(d.square().mean(-1, keepdim=True) + 1e-6) * after.double()
        x = want_r + d
        want = x * torch.rsqrt(x.square().mean(-1, keepdim=True) + 1e-5) * weight.double()
        # elements of a few units, float32 sums of up to 4,100 squares: relative errors of 1e-6 or so
        close(got, (want if picked is None else want[picked.long()]).float(), 2e-5, 2e-5)
        close(got_r, (x if picked is None else want_r).float(), 1e-5, 1e-5)


@pytest.mark.parametrize("dtype", [torch.float32, torch.bfloat16])
@pytest.mark.parametrize("t,h,n,top,how", [
    (1, 64, 3, 2, {}),
    (255, 260, 16, 2, {"scoring": "softmax_all", "groups": 4, "keep": 2, "group_score": "max"}),
    (256, 260, 16, 2, {"scoring": "softmax_all", "groups": 4, "keep": 2, "group_score": "max"}),
    (300, 2560, 16, 2, {}),
    (263, 128, 64, 8, {"scoring": "sigmoid", "groups": 8, "keep": 3}),
    (9, 128, 64, 64, {"scoring": "sigmoid"}),
    (257, 96, 20, 3, {"scoring": "softmax_all", "renormalise": True, "weight_scale": 2.5, "corrected": True}),
    (4, 128, 65, 4, {}),                              # beyond the lanes of a wave: the other kernel
    (258, 64, 1, 1, {"gate_row": True}),
    (2, 64, 6, 2, {"gate_row": True}),
])
def test_route_top(ops, dtype, t, h, n, top, how):
    how = dict(how)
    x = rnd(t, h, dtype=dtype, seed=1)
    router = rnd(n + int(how.get("gate_row", False)), h, seed=2, scale=2.0 * h ** -0.5)
    bias = rnd(n, seed=3)
    if how.pop("corrected", False):
        how["correction"] = 0.1 * rnd(n, seed=5)
    got = ops.route_top(x, router, bias, top, **how)
    want = R.route_top(x.double().float(), router, bias, top, **how)
    # scores of this size differ between two orders of float32 sums by 1e-6: where two lie closer the choice may differ
    same = (got[0].long() == want[0].long().to(DEV)).all(-1)
    assert same.float().mean() > 0.99
    close(got[1][same], want[1][same], 2e-5, 2e-5)
    assert (got[0].sort(-1).values.diff(dim=-1) > 0).all()   # an expert is chosen once
    if len(got) == 3:
        close(got[2], want[2], 2e-5, 2e-5)


def test_route_top_of_scores_that_are_no_numbers_stays_within_the_experts(ops):
    x = rnd(300, 64, seed=1)
    x[::3] = float("nan")
    x[1::7, 5] = float("inf")
    for n, top, how in ((16, 4, {}), (16, 2, {"scoring": "sigmoid", "groups": 4, "keep": 1}), (64, 64, {"scoring": "softmax_all"})):
        for rows in (x, x[:4].contiguous()):
            index, _ = ops.route_top(rows, rnd(n, 64, seed=2), None, top, **how)
            assert index.min() >= 0 and index.max() < n
            assert (index.sort(-1).values.diff(dim=-1) > 0).all()


@pytest.mark.parametrize("t", [3, 600])
@pytest.mark.parametrize("heads,width,pairs,in_stride,in_offset,out_stride,out_offset", [
    (4, 128, 64, 128, 0, 128, 0), (3, 64, 8, 192, 128, 96, 16), (2, 40, 0, 40, 0, 48, 8), (5, 24, 12, 24, 0, 24, 0),
])
@pytest.mark.parametrize("dtype,out_dtype", [(torch.bfloat16, torch.float32), (torch.bfloat16, torch.bfloat16), (torch.float32, torch.float32)])
def test_rotate_half(ops, t, heads, width, pairs, in_stride, in_offset, out_stride, out_offset, dtype, out_dtype):
    x = rnd(t, heads * in_stride, dtype=dtype, seed=1)
    freq = (1e4 ** -(torch.arange(pairs, dtype=torch.float32) / max(pairs, 1))).to(DEV) if pairs else None
    positions = (torch.arange(t, dtype=torch.int32, device=DEV) * 37 + 5)
    outs = [torch.full((t, heads * out_stride), 7.0, dtype=out_dtype, device=DEV) for _ in range(2)]
    ops.rotate_half(x, in_stride, in_offset, outs[0], out_stride, out_offset, heads, width, positions, freq, magnitude=1.25)
    R.rotate_half_copy(x, in_stride, in_offset, outs[1], out_stride, out_offset, heads, width, positions, freq, magnitude=1.25)
    tol = 1e-2 if out_dtype == torch.bfloat16 else 2e-5
    close(outs[0], outs[1], tol, tol)


@pytest.mark.parametrize("dtype", [torch.float32, torch.bfloat16])
@pytest.mark.parametrize("shape", [(1, 8), (3, 37), (1500, 1024)])
def test_squared_relu(ops, dtype, shape):
    x = rnd(*shape, dtype=dtype, seed=1)
    assert torch.equal(ops.unary_act(x, "relu2"), x.float().clamp(min=0).square().to(dtype))


# few rows in every kernel that takes them, tiles, and K that keeps to the two kernels; weight rows: a remainder of 16 goes there too
@pytest.mark.parametrize("n,k", [(16, 64), (400, 2560), (48, 128), (40, 192), (64, 96)])
def test_product_and_squared_relu_have_the_bits_of_the_two(ops, n, k):
    x, w = rnd(300, k, dtype=torch.bfloat16, seed=1), rnd(n, k, dtype=torch.bfloat16, seed=2, scale=k ** -0.5)
    for m in (1, 8, 9, 16, 17, 64, 65, 300):
        assert torch.equal(ops.act_linear(x[:m], w, "relu2"), ops.unary_act(ops.linear(x[:m], w), "relu2")), m


# weight rows: 512, 513, 768 and 769 tiles of 16 and a remainder; rows on both sides of 4, 8 and 16
@pytest.mark.parametrize("n", [8192, 8200, 12288, 12296])
@pytest.mark.parametrize("m", [1, 4, 5, 8, 9, 16])
def test_few_rows_at_the_edges_of_their_tiles(ops, m, n):
    x, w = rnd(m, 192, dtype=torch.bfloat16, seed=3), rnd(n, 192, dtype=torch.bfloat16, seed=4)
    want = x.double() @ w.double().T
    # float32 sums of 192 products; the result is not rounded further
    bound = 192 * 2.0 ** -24 * (x.double().abs() @ w.double().abs().T)
    assert ((ops.linear(x, w, out_f32=True).double() - want).abs() <= bound).all()


# K in eight planes: 128 and 129, 160 and 161 tiles of 16 and a remainder (a block has two, one, one, two), at the shortest K of the rule and
# in front of it; a part of the pairs of k-steps that is no multiple of the waves
@pytest.mark.parametrize("n", [2048, 2049, 2560, 2561])
@pytest.mark.parametrize("k", [9664, 9728, 12352])
def test_few_rows_in_planes_at_the_edges_of_their_tiles(ops, n, k):
    x, w = rnd(9, k, dtype=torch.bfloat16, seed=7), rnd(n, k, dtype=torch.bfloat16, seed=8, scale=k ** -0.5)
    for m in (1, 8, 9):
        planes = ops.linear_for_residual(x[:m], w)
        assert planes.shape == (8, m, n)
        # float32 sums of k products, as above
        bound = k * 2.0 ** -24 * (x[:m].double().abs() @ w.double().abs().T)
        assert ((planes.double().sum(0) - x[:m].double() @ w.double().T).abs() <= bound).all()


# tiles of eight gate and eight up rows or one of either: rows of K up to 4,096 and beyond, on both sides of 2 and 8 rows
@pytest.mark.parametrize("activation,limit", [("swiglu", 0.0), ("clamped", 0.9)])
@pytest.mark.parametrize("inter,k", [(8, 64), (20, 4096), (36, 4160)])
def test_gated_few_rows_at_the_edges_of_their_tiles(ops, inter, k, activation, limit):
    x, w = rnd(11, k, dtype=torch.bfloat16, seed=5), rnd(2 * inter, k, dtype=torch.bfloat16, seed=6, scale=2 * k ** -0.5)
    for m in (1, 2, 3, 8, 9, 11):
        both = (x[:m].double() @ w.double().T).float()
        want = ops.gated_act(both.to(torch.bfloat16), activation, limit)
        # both halves rounded to bfloat16 may fall on the other side of a tie: two units of 2^-8, as the result's own
        close(ops.gated_linear(x[:m], w, activation, limit), want, 2e-2, 2e-2)


@pytest.mark.parametrize("tokens", [1, 16, 17, 128, 129, 300])
@pytest.mark.parametrize("heads,n,k,in_stride,in_offset,out_stride,out_offset",
                         [(3, 4, 64, 64, 0, 4, 0), (2, 60, 128, 160, 24, 72, 8), (4, 384, 128, 192, 0, 448, 0),
                          (2, 132, 64, 72, 8, 136, 4), (5, 128, 384, 448, 64, 128, 0), (2, 64, 100, 104, 0, 64, 0), (2, 30, 64, 64, 0, 33, 3)])
def test_heads_linear_by_tiles(ops, tokens, heads, n, k, in_stride, in_offset, out_stride, out_offset):
    g = torch.Generator().manual_seed(tokens + n + k)
    x = torch.randn((tokens, heads * in_stride), generator=g).bfloat16()
    w = torch.randn((heads, n, k), generator=g).bfloat16()
    out = torch.full((tokens, heads * out_stride), 7.0).bfloat16()
    got = ops.heads_linear(x.cuda(), in_stride, in_offset, w.cuda(), out.cuda(), out_stride, out_offset).cpu().double()
    part = x.double().view(tokens, heads, in_stride)[:, :, in_offset: in_offset + k]
    want = torch.einsum("thk,hnk->thn", part, w.double())
    sizes = torch.einsum("thk,hnk->thn", part.abs(), w.double().abs())
    got = got.view(tokens, heads, out_stride)
    # k rounded additions in float32 and one rounding to bfloat16
    here = got[:, :, out_offset: out_offset + n]
    assert ((here - want).abs() <= k * 2.0 ** -24 * sizes + 2.0 ** -8 * want.abs() + 1e-30).all()
    outside = torch.ones(out_stride, dtype=torch.bool)
    outside[out_offset: out_offset + n] = False
    assert (got[:, :, outside] == 7.0).all()


def test_heads_wider_than_the_own_kernels_take_are_still_multiplied(ops):
    test_heads_linear_by_tiles(ops, 17, 1, 8, 16448, 16448, 0, 8, 0)


@pytest.mark.parametrize("tokens,heads,vdim", [(1, 1, 8), (3, 5, 24), (7, 3, 128), (33, 2, 512), (5, 2, 520), (65, 3, 40)])
@pytest.mark.parametrize("gate_dtype,out_dtype", [(torch.bfloat16, torch.bfloat16), (torch.float32, torch.float32), (torch.float32, torch.bfloat16)])
@pytest.mark.parametrize("kind", ["silu", "sigmoid"])
def test_read_out_norm_and_gate_in_pieces(ops, tokens, heads, vdim, gate_dtype, out_dtype, kind):
    g = torch.Generator().manual_seed(tokens + vdim)
    o, w = torch.randn((tokens, heads, vdim), generator=g), torch.randn(vdim, generator=g)
    wide = torch.randn((tokens, heads * vdim + 16), generator=g).to(gate_dtype)
    got = ops.delta_out(o.cuda(), w.cuda(), wide.cuda()[:, 8: 8 + heads * vdim], 1e-5, kind, out_dtype).double().cpu()
    z = wide[:, 8: 8 + heads * vdim].double().view(tokens, heads, vdim)
    act = torch.sigmoid(z) * (z if kind == "silu" else 1.0)
    want = (o.double() / (o.double().pow(2).mean(-1, keepdim=True) + 1e-5).sqrt() * w.double() * act).reshape(tokens, -1)
    # float32 on the way: a dozen roundings, the exponential of an argument up to 6; bfloat16: half of 2^-7
    rel = 40 * 2.0 ** -24 + (2.0 ** -8 if out_dtype == torch.bfloat16 else 0.0)
    assert ((got - want).abs() <= rel * want.abs() * 1.01 + 1e-30).all()


@pytest.mark.parametrize("tokens,width,first", [(1, 8, 8), (3, 40, 16), (65, 4096, 8), (5, 24, 4), (4, 30, 8)])
def test_sigmoid_gate_in_pieces(ops, tokens, width, first):
    g = torch.Generator().manual_seed(width)
    out = torch.randn((tokens, width), generator=g).bfloat16()
    wide = (3 * torch.randn((tokens, width + 24), generator=g)).bfloat16()
    got = ops.sigmoid_gate(out.cuda(), wide.cuda()[:, first: first + width]).double().cpu()
    want = out.double() * torch.sigmoid(wide[:, first: first + width].double())
    assert ((got - want).abs() <= (2.0 ** -8 * 1.01 + 40 * 2.0 ** -24) * want.abs()).all()
