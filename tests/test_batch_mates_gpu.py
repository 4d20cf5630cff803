"""What a request gets does not depend on what else is in its step: equal bits alone and beside others."""

import copy
import types

import pytest
import torch

from test_kernels_gpu import DEV, build_attention_case, rnd

pytestmark = pytest.mark.gpu


@pytest.fixture(scope="module")
def ops():
    from qwen3_runtime_amd.ops.hip import HipOps

    return HipOps()


def _part(ctx, cache, s, skip):
    """The step that holds nothing but the tokens of sequence ``s`` from its ``skip``-th on."""
    n, kv = ctx.q_lens_host[s] - skip, ctx.kv_lens_host[s]
    part, pages = copy.copy(ctx), copy.copy(cache)
    pages.group = copy.copy(cache.group)
    pages.group.block_table = cache.group.block_table[s: s + 1].contiguous()
    at = sum(ctx.q_lens_host[:s]) + skip
    part.num_tokens, part.num_seqs, part.q_lens_host, part.kv_lens_host = n, 1, [n], [kv]
    part.max_q_len, part.max_kv_len, part.scratch, part.groups = n, kv, {}, [pages.group]
    part.cu_q = torch.tensor([0, n], dtype=torch.int32, device=DEV)
    part.kv_lens, part.state_slots, part.first_span = ctx.kv_lens[s: s + 1], ctx.state_slots[s: s + 1], ctx.first_span[s: s + 1]
    part.positions, part.seq_of_token = ctx.positions[at: at + n].contiguous(), torch.zeros(n, dtype=torch.int32, device=DEV)
    return part, pages, slice(at, at + n)


@pytest.mark.parametrize("nq,nkv,d,more", [(4, 2, 128, {}), (8, 8, 32, {"window": 40}), (5, 1, 256, {"window": 70, "keep_first": 21})])
def test_float32_attention(ops, nq, nkv, d, more):
    """Many sequences, or one; a prompt in one step, or most of it in a step of its own."""
    seqs = [(1, 300), (40, 131), (1, 17), (90, 90)] + [(3, 64)] * 200
    q, cache, ctx = build_attention_case(seqs, nq, nkv, d, 16, torch.float32, window=more.get("window"), poison=True)
    attend = lambda q, cache, ctx: ops.paged_attention(q, cache, ctx, nq, nkv, d, d ** -0.5, more.get("window"),  # noqa: E731
                                                       keep_first=more.get("keep_first", 0))
    whole = attend(q, cache, ctx)
    assert torch.isfinite(whole).all()
    for s, skip in ((0, 0), (1, 0), (2, 0), (3, 0), (3, 7), (150, 0)):
        part, pages, rows = _part(ctx, cache, s, skip)
        assert torch.equal(attend(q[rows].contiguous(), pages, part), whole[rows]), (s, skip)


@pytest.mark.parametrize("dim,vdim", [(64, 32), (128, 40), (200, 16)])
@pytest.mark.parametrize("lengths", [(1, 1, 300, 1), (63, 64, 65, 127, 128, 1), (2,) * 40 + (133,), (130,) * 160])
def test_retention(ops, dim, vdim, lengths):
    heads, t = 3, sum(lengths)
    qkv, state = rnd(t, 2 * heads * dim + heads * vdim, seed=1), rnd(len(lengths), heads, vdim, dim, seed=2)
    decay = torch.tensor([0.9, 0.99, 0.5], device=DEV)

    def run(lengths, qkv, slots, on_host):
        cu = torch.tensor([0, *torch.tensor(lengths).cumsum(0).tolist()], dtype=torch.int32, device=DEV)
        ctx = types.SimpleNamespace(num_tokens=sum(lengths), num_seqs=len(lengths), cu_q=cu,
                                    state_slots=torch.tensor(slots, dtype=torch.int32, device=DEV))
        if on_host:  # without its lengths on the host a step launches both forms
            ctx.q_lens_host = list(lengths)
        after = state.clone()
        return ops.retention_rule(ctx, qkv, decay, after, heads, dim, vdim), after

    whole, after = run(lengths, qkv, range(len(lengths)), True)
    assert all(torch.equal(a, b) for a, b in zip(run(lengths, qkv, range(len(lengths)), False), (whole, after)))
    at = 0
    for s, n in enumerate(lengths[:6]):
        got, own = run((n,), qkv[at: at + n].contiguous(), [s], True)
        assert torch.equal(got, whole[at: at + n]) and torch.equal(own[s], after[s]), (s, n)
        at += n


@pytest.mark.parametrize("dtype", [torch.float32, torch.bfloat16])
@pytest.mark.parametrize("hidden", [64, 1000, 2560, 5120])
@pytest.mark.parametrize("how", [{"scoring": "sigmoid"}, {"scoring": "softmax_all", "groups": 4, "keep": 2, "group_score": "max"}, {}])
def test_router_and_its_gate(ops, dtype, hidden, how):
    """Steps of many tokens share the router's rows among eight; a token's choice, weights and gate are the same."""
    x, router = rnd(805, hidden, dtype=dtype, seed=1), rnd(17, hidden, seed=2, scale=2.0 * hidden ** -0.5)
    whole = ops.route_top(x, router, None, 3, gate_row=True, **how)
    for a, b in ((0, 1), (5, 13), (300, 805)):
        part = ops.route_top(x[a:b].contiguous(), router, None, 3, gate_row=True, **how)
        assert all(torch.equal(p, w[a:b]) for p, w in zip(part, whole))


@pytest.mark.parametrize("hidden", [64, 1000, 2048, 2560, 4096, 4100])
@pytest.mark.parametrize("planes", [1, 2, 4])
def test_norm_behind_a_sublayer(ops, hidden, planes):
    """Steps of many tokens take a quarter of the threads a row; a token's sums are the same."""
    t = 700
    y = rnd(t, hidden, seed=1) if planes == 1 else rnd(planes, t, hidden, seed=1)
    residual, after, weight = rnd(t, hidden, seed=2), rnd(hidden, seed=3), rnd(hidden, seed=4)
    norm = lambda r, y, **more: ops.add_rmsnorm(r, y, weight, 1e-5, torch.float32, delta_norm=(after, 1e-6), **more)  # noqa: E731
    whole_r = residual.clone()
    whole = norm(whole_r, y)
    for a, b in ((0, 1), (5, 13), (100, 600)):
        part_r = residual[a:b].clone()
        part = norm(part_r, y[..., a:b, :].contiguous())
        assert torch.equal(part, whole[a:b]) and torch.equal(part_r, whole_r[a:b])
    rows = torch.tensor([3, 699, 4], dtype=torch.int32, device=DEV)
    assert torch.equal(norm(residual.clone(), y, rows=rows), whole[rows.long()])
