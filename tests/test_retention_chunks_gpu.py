"""Retention over prompts by chunks of tokens: against the recurrence in float64, at the edges of chunks, heads and columns."""

import math
import types

import pytest
import torch

pytestmark = pytest.mark.gpu
EPS = 2.0 ** -24


@pytest.fixture(scope="module")
def ops():
    from qwen3_runtime_amd.ops.hip import HipOps
    return HipOps()


def _draw(lengths, heads, dim, vdim, decay, seed=0):
    g = torch.Generator().manual_seed(seed)
    t = sum(lengths)
    qkv = torch.randn((t, 2 * heads * dim + heads * vdim), generator=g)
    slots = torch.randperm(len(lengths) + 2, generator=g)[:len(lengths)].to(torch.int32)
    state = torch.randn((len(lengths) + 2, heads, vdim, dim), generator=g)
    return qkv, torch.tensor([decay[h % len(decay)] for h in range(heads)]), state, slots


def _recurrence(lengths, qkv, decay, state, slots, heads, dim, vdim):
    """Read-outs and states in float64, and for both the same sums over sizes (what rounding is relative to)."""
    t = qkv.shape[0]
    q, k, v = (x.double() for x in qkv.split([heads * dim, heads * dim, heads * vdim], 1))
    q, k, v = q.view(t, heads, dim), k.view(t, heads, dim), v.view(t, heads, vdim)
    state, out = state.double().clone(), torch.empty((t, heads, vdim), dtype=torch.float64)
    sizes, out_sizes = state.abs(), torch.empty_like(out)
    d, at = decay.double()[:, None, None], 0
    for n, slot in zip(lengths, slots.tolist()):
        for i in range(at, at + n):
            state[slot] = d * state[slot] + v[i][:, :, None] * k[i][:, None, :]
            sizes[slot] = d.abs() * sizes[slot] + v[i].abs()[:, :, None] * k[i].abs()[:, None, :]
            out[i] = (state[slot] * q[i][:, None, :]).sum(-1)
            out_sizes[i] = (sizes[slot] * q[i].abs()[:, None, :]).sum(-1)
        at += n
    return out, out_sizes, state, sizes


def _run(ops, lengths, qkv, decay, state, slots, heads, dim, vdim):
    cu = torch.tensor([0, *torch.tensor(lengths).cumsum(0).tolist()], dtype=torch.int32)
    ctx = types.SimpleNamespace(num_tokens=sum(lengths), num_seqs=len(lengths), cu_q=cu.cuda(), state_slots=slots.cuda())
    state = state.cuda()
    return ops.retention_rule(ctx, qkv.cuda(), decay.cuda(), state, heads, dim, vdim).cpu(), state.cpu()


@pytest.mark.parametrize("dim,vdim,heads", [(4, 1, 2), (60, 16, 3), (64, 40, 2), (68, 17, 2), (128, 128, 4), (132, 16, 1), (256, 33, 2)])
@pytest.mark.parametrize("lengths", [(3,), (31,), (32,), (33, 1, 64), (100, 7)])
@pytest.mark.parametrize("decay", [(0.9, 0.5), (1.0, 0.0), (-0.7, 0.999)])
def test_chunks_match_the_recurrence(ops, dim, vdim, heads, lengths, decay):
    qkv, d, state, slots = _draw(lengths, heads, dim, vdim, decay)
    out, out_sizes, states, sizes = _recurrence(lengths, qkv, d, state, slots, heads, dim, vdim)
    got, after = _run(ops, lengths, qkv, d, state, slots, heads, dim, vdim)
    # a term takes part in at most `longest` + dim additions and passes `longest` decays, each one rounding
    steps = 2 * max(lengths) + dim + 8
    assert ((got.double() - out).abs() <= steps * EPS * out_sizes).all()
    assert ((after.double() - states).abs() <= steps * EPS * sizes).all()


@pytest.fixture(scope="module")
def chunking():
    """Spans of any length by chunks."""
    from qwen3_runtime_amd.ops.hip import HipOps

    ops = HipOps()
    ops.retention_chunk_min_tokens = 1
    return ops


@pytest.mark.parametrize("lengths,heads,dim,vdim", [((1,), 1, 4, 1), ((31,), 3, 60, 16), ((32, 33, 2), 2, 68, 17), ((65, 3), 2, 256, 33),
                                                    ((33, 1, 64, 97) * 3, 4, 68, 128), ((33, 1, 64, 97) * 3, 9, 60, 128)])
def test_every_form_of_the_chunks_matches_the_recurrence(chunking, lengths, heads, dim, vdim):
    """Spans of any length by chunks, in launches of few blocks and of many (the last two)."""
    decay = (0.9, -0.7, 1.0, 0.5)
    qkv, d, state, slots = _draw(lengths, heads, dim, vdim, decay)
    out, out_sizes, states, sizes = _recurrence(lengths, qkv, d, state, slots, heads, dim, vdim)
    got, after = _run(chunking, lengths, qkv, d, state, slots, heads, dim, vdim)
    steps = 2 * max(lengths) + dim + 8
    assert ((got.double() - out).abs() <= steps * EPS * out_sizes).all()
    assert ((after.double() - states).abs() <= steps * EPS * sizes).all()


@pytest.mark.parametrize("which", ["k", "v", "q"])
@pytest.mark.parametrize("value", [float("inf"), float("nan"), 1e30])
def test_a_value_that_is_not_finite_stays_behind_its_token(ops, which, value):
    heads, dim, vdim, lengths, at = 2, 64, 32, (70,), 41
    qkv, d, state, slots = _draw(lengths, heads, dim, vdim, (0.9, 0.5))
    qkv[at, {"q": 3, "k": heads * dim + 3, "v": 2 * heads * dim + 3}[which]] = value
    out, out_sizes, _, _ = _recurrence(lengths, qkv, d, state, slots, heads, dim, vdim)
    got, _ = _run(ops, lengths, qkv, d, state, slots, heads, dim, vdim)
    steps = 2 * max(lengths) + dim + 8
    assert ((got.double() - out).abs() <= steps * EPS * out_sizes)[:at].all()
    fine = torch.isfinite(out) & (out.abs() < 3e38)
    assert (torch.isfinite(got) == fine).all()
    assert ((got.double() - out).abs() <= steps * EPS * out_sizes)[fine].all()


@pytest.mark.parametrize("size", [1e30, 3e37, float("inf")])
@pytest.mark.parametrize("where", ["state", "k", "v"])
def test_what_a_large_state_holds_decays_as_in_the_recurrence(chunking, size, where):
    """Read-outs and states that the recurrence keeps finite are finite and right, and one that became infinite stays so."""
    heads, dim, vdim, lengths = 4, 64, 20, (80,)
    qkv, d, state, slots = _draw(lengths, heads, dim, vdim, (0.0, 0.1, 0.5, 0.999))
    qkv[:, : heads * dim] *= 100.0
    if where == "state":
        state[:, :, :, 2] *= size
    else:
        qkv[9, {"k": slice(heads * dim + 2, 2 * heads * dim, dim), "v": slice(2 * heads * dim + 2, None, vdim)}[where]] *= size
    out, out_sizes, _, _ = _recurrence(lengths, qkv, d, state, slots, heads, dim, vdim)
    got, after = _run(chunking, lengths, qkv, d, state, slots, heads, dim, vdim)
    steps = 2 * max(lengths) + dim + 8
    fine = torch.isfinite(out) & (out_sizes < 1e37)
    if not math.isinf(size):
        assert fine.float().mean() > 0.5
    assert ((got.double() - out).abs() <= steps * EPS * out_sizes + 1e-30)[fine].all()
    walked = state[slots.long()].clone()[0]
    q, k, v = qkv.split([heads * dim, heads * dim, heads * vdim], 1)
    for i in range(80):
        walked = d[:, None, None] * walked + v[i].view(heads, vdim, 1) * k[i].view(heads, 1, dim)
    last = after[int(slots[0])]
    assert torch.equal(torch.isnan(last), torch.isnan(walked))
    assert torch.equal(last[torch.isinf(walked)], walked[torch.isinf(walked)])


@pytest.mark.parametrize("which", ["k", "v", "q"])
@pytest.mark.parametrize("value", [float("inf"), float("nan"), 1e30])
def test_a_value_that_is_not_finite_stays_behind_its_token_in_chunks(chunking, which, value):
    test_a_value_that_is_not_finite_stays_behind_its_token(chunking, which, value)
