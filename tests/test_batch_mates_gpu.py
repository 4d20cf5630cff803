"""What a request gets does not depend on what else is in its step: equal bits alone and beside others."""

import copy

import pytest
import torch

from test_kernels_gpu import DEV, build_attention_case

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
