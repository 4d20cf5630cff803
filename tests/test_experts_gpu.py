"""The routed experts' MFMA kernels against the plain experts in float64, in both forms (a stream of the
weights, tiles), at the edges of their groups of 16 and 128 pairs."""

import pytest
import torch

from test_kernels_gpu import DEV, close, rnd

pytestmark = pytest.mark.gpu


@pytest.fixture()
def ops():
    from qwen3_runtime_amd.ops.hip import HipOps

    return HipOps()


def plain(x, gate_up, down, index, weight, activation, limit, on_input):
    """float64 [top, T, H]; the activations rounded to bfloat16 between the two products."""
    t, top = index.shape
    x, gate_up, down, weight = x.double(), gate_up.double(), down.double(), weight.double()
    out = torch.zeros(top, t, x.shape[1], dtype=torch.float64, device=x.device)
    for i in range(t):
        for j in range(top):
            e = int(index[i, j])
            by = weight[i, j] if on_input else 1.0
            z = gate_up[e] @ x[i] * by
            if activation == "relu2":
                a = z.clamp(min=0).square()
            else:
                g, u = z.chunk(2)
                if activation == "clamped":
                    g, u = g.clamp(max=limit), u.clamp(-limit, limit)
                    a = g * torch.sigmoid(1.702 * g) * (u + 1)
                else:
                    a = g * torch.sigmoid(g) * u
            out[j, i] = down[e] @ a.bfloat16().double() * (1.0 if on_input else weight[i, j])
    return out


@pytest.mark.parametrize("form", ["stream", "tiles"])
@pytest.mark.parametrize("t,top,n,h,inter,skew,activation,on_input", [
    (1, 2, 16, 128, 64, None, "swiglu", False),     # fewer pairs than experts
    (5, 3, 4, 192, 128, None, "clamped", False),    # K of three pieces of 64, one wave without any
    (17, 1, 3, 64, 192, 0, "swiglu", True),         # 17 pairs of one expert: two groups of 16; experts without a pair
    (40, 2, 5, 128, 64, None, "relu2", False),
    (129, 1, 2, 64, 64, 1, "swiglu", False),        # 129 pairs of one expert: two tiles, the second of one pair
    (150, 8, 64, 128, 128, None, "swiglu", False),
])
def test_experts_against_float64(ops, form, t, top, n, h, inter, skew, activation, on_input):
    ops.experts_tile_pairs_per_expert = 0 if form == "tiles" else 1 << 20
    gated = activation != "relu2"
    x = rnd(t, h, dtype=torch.bfloat16, seed=1)
    gate_up = rnd(n, (2 if gated else 1) * inter, h, dtype=torch.bfloat16, scale=h ** -0.5, seed=2)
    down = rnd(n, h, inter, dtype=torch.bfloat16, scale=inter ** -0.5, seed=3)
    scores = rnd(t, n, seed=4)
    if skew is not None:
        scores[:, skew] += 100.0
    weight, index = scores.topk(top, -1)
    weight, index = torch.softmax(weight, -1).contiguous(), index.int().contiguous()
    want = plain(x, gate_up, down, index, weight, activation, 2.0, on_input)
    got = ops.moe_for_residual(x, gate_up, down, index, weight, activation, 2.0, on_input)
    # an activation (about one in size) that float32 sums bring to the other side of a bfloat16 boundary is 2^-8 off:
    # times a weight of size inter^-0.5, and few of an output's terms are
    close(got, want.float(), 4e-3, 4e-3)
    close(ops.moe_swiglu(x, gate_up, down, index, weight, activation, 2.0, weight_on_input=on_input), want.sum(0).float(), 8e-3, 8e-3)


def test_widths_that_whole_lines_do_not_fit_keep_the_general_form(ops):
    x, gate_up, down = (rnd(*s, dtype=torch.bfloat16, scale=0.1) for s in ((3, 96), (4, 80, 96), (4, 96, 40)))
    index = torch.tensor([[0, 3], [1, 0], [2, 1]], dtype=torch.int32, device=DEV)
    weight = torch.full((3, 2), 0.5, device=DEV)
    assert ops.moe_for_residual(x, gate_up, down, index, weight) is None
    want = plain(x, gate_up, down, index, weight, "swiglu", 0.0, False).sum(0)
    close(ops.moe_swiglu(x, gate_up, down, index, weight), want.float(), 1e-3, 1e-3)


@pytest.mark.parametrize("which,t", [("x", 3), ("x", 70), ("gate_up", 3), ("down", 3)])
def test_operands_that_begin_between_16_bytes_keep_the_general_form(ops, which, t):
    def at_8_bytes(a):
        room = torch.empty(a.numel() + 4, dtype=a.dtype, device=DEV)
        room[4:].copy_(a.reshape(-1))
        return room[4:].view(a.shape)

    x, gate_up, down = (rnd(*s, dtype=torch.bfloat16, scale=0.1) for s in ((t, 128), (4, 128, 128), (4, 128, 64)))
    scores = rnd(t, 4, seed=4)
    weight, index = scores.topk(2, -1)
    weight, index = torch.softmax(weight, -1).contiguous(), index.int().contiguous()
    want = plain(x, gate_up, down, index, weight, "swiglu", 0.0, False).sum(0)
    moved = {"x": x, "gate_up": gate_up, "down": down}
    moved[which] = at_8_bytes(moved[which])
    assert moved[which].is_contiguous() and moved[which].data_ptr() % 16 == 8
    assert ops.moe_for_residual(moved["x"], moved["gate_up"], moved["down"], index, weight) is None
    close(ops.moe_swiglu(moved["x"], moved["gate_up"], moved["down"], index, weight), want.float(), 1e-3, 1e-3)


@pytest.mark.parametrize("tokens", [1, 8, 40])
@pytest.mark.parametrize("experts,top", [(16, 8), (16, 12), (64, 64)])
def test_any_number_of_experts_a_token_beside_a_shared_expert(ops, tokens, experts, top):
    """The feed-forward part's result goes into the next norm as it is, however many experts a token has."""
    from types import SimpleNamespace

    from test_zisedra import DictFetch

    from qwen3_runtime_amd.parts.moe import RoutedSwiGLU

    width, inner, shared = 128, 64, 128
    names = {"router": "r", "gate": "e{e}.gate", "up": "e{e}.up", "down": "e{e}.down",
             "shared_gate": "s.gate", "shared_up": "s.up", "shared_down": "s.down"}
    w = {"r": rnd(experts, width, scale=0.3), "s.gate": rnd(shared, width, seed=2, scale=0.1), "s.up": rnd(shared, width, seed=3, scale=0.1),
         "s.down": rnd(width, shared, seed=4, scale=0.1)}
    for e in range(experts):
        w[f"e{e}.gate"], w[f"e{e}.up"], w[f"e{e}.down"] = (rnd(*s, seed=10 * i + e, scale=0.1)
                                                            for i, s in ((1, (inner, width)), (9, (inner, width)), (17, (width, inner))))
    w = {n: a.cpu().bfloat16().float() for n, a in w.items()}
    part = RoutedSwiGLU(width, inner, experts, top, router_bias=False, scoring="sigmoid", shared_size=shared, tensors=names)
    part.load(DictFetch(w, DEV, torch.bfloat16))
    x = rnd(tokens, width, dtype=torch.bfloat16, seed=5)
    y = part.forward(SimpleNamespace(ops=ops, dtype=torch.bfloat16), x)
    residual = torch.zeros(tokens, width, device=DEV)
    ops.add_rmsnorm(residual, y, torch.ones(width, device=DEV), 1e-6, torch.float32)
    dev = {n: a.to(DEV).double() for n, a in w.items()}
    weight, index = torch.sigmoid(x.double() @ dev["r"].T).topk(top, -1)
    gate_up = torch.stack([torch.cat([dev[f"e{e}.gate"], dev[f"e{e}.up"]]) for e in range(experts)])
    down = torch.stack([dev[f"e{e}.down"] for e in range(experts)])
    want = plain(x, gate_up, down, index, weight, "swiglu", 0.0, False).sum(0)
    g = x.double() @ dev["s.gate"].T
    want += (g * torch.sigmoid(g) * (x.double() @ dev["s.up"].T)).bfloat16().double() @ dev["s.down"].T
    # activations of up to a few units that fall on the other side of a bfloat16 boundary, times weights of 0.1, and sums of
    # `top` such outputs; a choice that falls the other way in float32 moves a token
    bad = ((residual.double() - want).abs() > 2e-2 + 2e-2 * want.abs()).any(-1)
    assert int(bad.sum()) <= tokens // 10
