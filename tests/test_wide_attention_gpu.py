"""Prompt portions with heads wider than 256 (rows of a latent): the kernel whose eight waves share keys and
values through LDS, at the edges of its tiles of 128 rows and blocks of 32 keys."""

import copy
import math

import pytest
import torch

from plain import ops_ref as R
from test_kernels_gpu import DEV, build_attention_case, close, rnd

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


@pytest.mark.parametrize("d,dv,nq,nkv,splits,more", [
    (448, 448, 32, 1, None, {"softcap": 3.0}),
    (448, 448, 16, 1, 3, {"softcap": 3.0, "sink": True}),
    (320, 320, 16, 1, None, {"chunk": 40}),
    (320, 320, 16, 1, 2, {"chunk": 40, "gate": True}),
    (448, 448, 8, 1, None, {"sink": True, "gate": True}),
    (448, 448, 8, 1, None, {"turn": True}),
    (320, 320, 8, 1, 2, {"turn": True, "sink": True}),
    (320, 64, 32, 1, None, {}),                       # values narrower than the loads asked for ahead
    (320, 64, 12, 3, 2, {"window": 50, "gate": True}),
    (64, 320, 16, 2, None, {"sink": True}),           # and keys
    (64, 320, 16, 2, 2, {"turn": True}),
])
def test_options_of_portions_with_wide_heads(d, dv, nq, nkv, splits, more):
    from qwen3_runtime_amd.ops.hip import HipOps

    ops, more = HipOps(), dict(more)
    window = more.pop("window", None)
    q, cache, ctx = build_attention_case([(70, 97), (9, 9), (1, 130), (33, 64)], nq, nkv, d, 16, torch.bfloat16, window=window, poison=dv == d)
    if dv != d:
        cache.v = rnd(cache.v.shape[0], nkv, dv, 16, dtype=torch.bfloat16, seed=7)
    if splits:
        ctx.scratch["attn_splits"] = splits
    if more.pop("gate", False):
        more["gate"] = rnd(ctx.num_tokens, nq * dv, dtype=torch.bfloat16, seed=9)
    if more.pop("turn", False):
        more["value_turn"] = (1e3 ** -(torch.arange(dv // 2, dtype=torch.float32, device=DEV) / (dv // 2)), "turned")
    scale = 1.0 / math.sqrt(d)
    want = R.paged_attention(q, cache.k, cache.v, ctx.cu_q.cpu(), ctx.kv_lens.cpu(), cache.group.block_table, 16, nq, nkv, d,
                             scale, window, value_dim=dv, **more)
    got = ops.paged_attention(q, cache, ctx, nq, nkv, d, scale, window, value_dim=dv, **more)
    assert next(p for k, p in ctx.scratch.items() if k[0] == "attn_plan")[3] == 3   # by the kernel that this file is about
    # as above; a turned output is made of two of them
    close(got, want, 2e-2, 2e-2)


@pytest.mark.parametrize("value", [float("inf"), float("-inf"), float("nan")])
@pytest.mark.parametrize("d,nq,splits,more", [(448, 32, None, {}), (448, 4, 3, {"window": 40}), (320, 16, 2, {"chunk": 32}),
                                              (320, 5, None, {"window": 23, "turn": True, "sink": True, "softcap": 3.0, "gate": True}),
                                              (512, 2, 2, {"turn": True, "sink": True})])
def test_a_token_takes_nothing_from_keys_it_does_not_see(value, d, nq, splits, more):
    """A value and a key of one token that are not finite: tokens that do not see it are as they are without it."""
    from qwen3_runtime_amd.ops.hip import HipOps

    ops, more, n = HipOps(), dict(more), 75
    window = more.pop("window", None)
    q, cache, ctx = build_attention_case([(n, n), (9, n)], nq, 1, d, 16, torch.bfloat16)
    if splits:
        ctx.scratch["attn_splits"] = splits
    if more.pop("gate", False):
        more["gate"] = rnd(ctx.num_tokens, nq * d, dtype=torch.bfloat16, seed=9)
    if more.pop("turn", False):
        more["value_turn"] = (1e3 ** -(torch.arange(d // 2, dtype=torch.float32, device=DEV) / (d // 2)), "turned")
    attend = lambda cache: ops.paged_attention(q, cache, ctx, nq, 1, d, d ** -0.5, window, **more)  # noqa: E731
    want, pos = attend(cache), torch.cat([torch.arange(n), torch.arange(n - 9, n)]).to(DEV)
    assert next(p for k, p in ctx.scratch.items() if k[0] == "attn_plan")[3] == 3
    assert torch.isfinite(want).all()
    for at in (0, 3, 31, 37, 74):
        sees = pos >= at
        if window:
            sees &= pos - at < window
        if "chunk" in more:
            sees &= pos // 32 == at // 32
        for stream in ("v", "k"):
            odd = copy.copy(cache)
            odd.k, odd.v = cache.k.clone(), cache.v.clone()
            for s in (0, 1):
                page, off = int(cache.group.block_table[s, at // 16]), at % 16
                if stream == "v":
                    odd.v[page, :, d - 1, off] = value
                else:
                    odd.k[page, :, off, 0] = value
            # one rounding to bfloat16 of results whose probabilities were rounded to it, or were not
            close(attend(odd)[~sees], want[~sees], 2e-2, 2e-2)


@pytest.mark.parametrize("d,nq,nkv,seqs,splits,more", [
    (448, 32, 1, [(1, 1), (1, 33), (1, 96)], None, {}),              # one block of keys a part; a sequence with fewer of them
    (448, 24, 1, [(1, 64)], None, {}),                               # 24 rows: the second wave's tile half full
    (320, 8, 2, [(1, 300), (1, 77)], None, {"window": 50}),
    (320, 72, 2, [(1, 300), (1, 77)], 1, {"window": 50, "keep_first": 37}),  # three waves, one without rows; kept keys: two blocks more
    (512, 16, 1, [(1, 1030), (2, 40)], None, {"sink": True}),        # the most LDS
    (512, 16, 1, [(1, 200)], 1, {"chunk": 40}),
])
def test_decoded_tokens_with_wide_heads(d, nq, nkv, seqs, splits, more):
    """The kernel that keeps the queries of heads wider than 256 in LDS, against the oracle."""
    from qwen3_runtime_amd.ops.hip import HipOps

    ops, more = HipOps(), dict(more)
    window = more.pop("window", None)
    q, cache, ctx = build_attention_case(seqs, nq, nkv, d, 16, torch.bfloat16, poison=True)
    if splits:
        ctx.scratch["attn_splits"] = splits
    scale = 1.0 / math.sqrt(d)
    want = R.paged_attention(q, cache.k, cache.v, ctx.cu_q.cpu(), ctx.kv_lens.cpu(), cache.group.block_table, 16, nq, nkv, d,
                             scale, window, **more)
    got = ops.paged_attention(q, cache, ctx, nq, nkv, d, scale, window, **more)
    assert next(p for k, p in ctx.scratch.items() if k[0] == "attn_plan")[3] != 3   # not by the kernel of the portions
    close(got, want, 2e-2, 2e-2)    # as above
