"""The row block that layers of fewer than 32 experts get."""
import pytest


@pytest.mark.parametrize("tokens,topk,experts,expected", [
    (128, 2, 8, 64),       # 32 rows per expert
    (132, 2, 8, 64),       # 33: one block of 64 still holds an expert
    (200, 2, 8, 64),       # 50
    (204, 2, 8, 128),      # 51
    (387, 4, 31, 64),      # 49.9
    (400, 4, 32, 128),     # 50, but enough experts for loads to differ
])
def test_few_experts(tokens, topk, experts, expected):
    from pyhip_amd.fused_moe import pick_block_m
    assert pick_block_m(tokens, topk, experts) == expected


def test_bf16_activations_keep_their_rule():
    from pyhip_amd import _lib
    lib = _lib.load()
    assert [lib.pyhip_moe_pick_block_m(t, 2, 8, 4096, 1) for t in (16, 64, 128, 200, 4096)] == [16, 32, 64, 64, 64]
