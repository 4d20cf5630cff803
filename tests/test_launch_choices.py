"""How launches are cut: the choices that go by measured lines, where the measurements lie."""

import pytest

from qwen3_runtime_amd.ops.hip import HipOps


@pytest.mark.parametrize("experts,inter,pairs", [(16, 1536, 15), (64, 768, 9), (8, 1024, 32), (4, 512, 32), (1024, 64, 9), (1, 64, 32)])
def test_pairs_an_expert_from_which_tiles_are_taken(experts, inter, pairs):
    assert HipOps.choose_experts_tile_pairs(experts, inter) == pairs


@pytest.mark.parametrize("d", [320, 448])
def test_parts_of_the_keys_of_portions_with_wide_heads(d):
    def parts(*seqs):
        walks = [((kv - n + (min(32 * n, r + 128) - 1) // 32) >> 5) + 1 for n, kv in seqs for r in range(0, 32 * n, 128)]
        return HipOps.choose_wide_splits(walks, 1, 4.0 * sum(n for n, _ in seqs) * 32 * d)

    assert parts((300, 300), (300, 300), (300, 300)) == parts((1000, 1000)) == parts(*[(150, 150)] * 5) == 1
    assert parts((1000, 3000), *[(1, 200)] * 8) == 1
    assert 3 <= parts((200, 4000)) <= 6 and parts((33, 8000)) >= 10
