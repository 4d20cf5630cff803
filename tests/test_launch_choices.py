"""How launches are cut: the choices that go by measured lines, where the measurements lie."""

import pytest

from qwen3_runtime_amd.ops.hip import HipOps


@pytest.mark.parametrize("sequences,keys,parts", [
    (1, 128, (1, 1)), (1, 200, (1, 1)), (8, 128, (1, 1)), (16, 200, (1, 1)), (48, 320, (1, 1)),     # the merge costs more than it saves
    (1, 320, (4, 8)), (6, 320, (4, 5)), (1, 640, (8, 16)), (1, 1025, (16, 16)), (8, 1025, (4, 4)),  # few sequences: many units
    (12, 2100, (2, 5)), (24, 2100, (4, 4)), (32, 2049, (1, 1)), (40, 2100, (4, 4)),
])
def test_parts_of_decoded_tokens_keys(sequences, keys, parts):
    assert parts[0] <= HipOps.choose_decode_splits(sequences, 8, keys) <= parts[1]


# a captured step is cut by its bucket: twice as many parts where one block falls to nearly every unit and the bucket has 256 keys for each
@pytest.mark.parametrize("sequences,keys,parts", [(7, 1025, 8), (8, 513, 4), (8, 1024, 4), (8, 1025, 8), (8, 2047, 8), (8, 2054, 8), (12, 2054, 5), (16, 1025, 4),
                                                  (16, 600, 4), (32, 2054, 1)])
def test_parts_of_a_captured_step(sequences, keys, parts):
    from qwen3_runtime_amd.engine.graph import DecodeGraph

    assert HipOps.choose_decode_splits(sequences, 8, DecodeGraph.key_for(sequences, keys, True)[1]) == parts


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


@pytest.mark.parametrize("sequences,keys,parts", [
    (8, 64, 1), (8, 65, 3), (8, 300, 10), (8, 512, 16), (8, 513, 9), (30, 128, 4), (1, 1024, 32), (1, 1025, 17), (16, 256, 8), (17, 256, 4),
    (8, 1029, 17), (300, 2000, 1),
])
def test_parts_of_the_keys_of_decoded_tokens_with_wide_heads(sequences, keys, parts):
    assert HipOps.choose_splits(sequences, 1, keys, 448) == parts
