"""Prompt portions with heads wider than 256 (rows of a latent): the kernel whose eight waves share keys and
values through LDS, at the edges of its tiles of 128 rows and blocks of 32 keys."""

import math

import pytest
import torch

from plain import ops_ref as R
from test_kernels_gpu import build_attention_case, close

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("d,seqs,nq,ps,window,splits", [
    (448, [(5, 5), (17, 40), (1, 33)], 32, 16, None, None),      # 160 and 544 rows; a decoded token beside them
    (448, [(70, 97)], 4, 8, None, None),
    (448, [(130, 131)], 2, 24, None, 3),                         # pages that are no power of two; keys over three blocks
    (320, [(64, 200), (9, 300)], 16, 16, 50, None),              # a window whose first pages are gone
    (320, [(40, 64)], 3, 32, None, None),
    (512, [(33, 96), (8, 8)], 16, 16, None, 2),
])
def test_portions_with_wide_heads(d, seqs, nq, ps, window, splits):
    from qwen3_runtime_amd.ops.hip import HipOps

    ops = HipOps()
    q, cache, ctx = build_attention_case(seqs, nq, 1, d, ps, torch.bfloat16, window=window, poison=True)
    if splits:
        ctx.scratch["attn_splits"] = splits
    scale = 1.0 / math.sqrt(d)
    want = R.paged_attention(q, cache.k, cache.v, ctx.cu_q.cpu(), ctx.kv_lens.cpu(), cache.group.block_table, ps, nq, 1, d,
                             scale, window)
    if window:
        table = cache.group.block_table.clone()
        for s, (ql, kv) in enumerate(seqs):
            for p in range(table.shape[1]):
                if (p + 1) * ps <= kv - ql - window + 1:
                    table[s, p] = -1
        cache.group.block_table = table
    got = ops.paged_attention(q, cache, ctx, nq, 1, d, scale, window)
    # as for the other head sizes: probabilities rounded to bfloat16, values of size 3
    close(got, want, 2e-2, 2e-2)


@pytest.mark.parametrize("d", [320, 448])
def test_how_many_parts_the_keys_of_portions_with_wide_heads_are_cut_into(d):
    from qwen3_runtime_amd.ops.hip import HipOps

    def parts(*seqs):
        walks = [((kv - n + (min(32 * n, r + 128) - 1) // 32) >> 5) + 1 for n, kv in seqs for r in range(0, 32 * n, 128)]
        return HipOps.choose_wide_splits(walks, 1, 4.0 * sum(n for n, _ in seqs) * 32 * d)

    assert parts((300, 300), (300, 300), (300, 300)) == parts((1000, 1000)) == parts(*[(150, 150)] * 5) == 1
    assert parts((1000, 3000), *[(1, 200)] * 8) == 1
    assert 3 <= parts((200, 4000)) <= 6 and parts((33, 8000)) >= 10
