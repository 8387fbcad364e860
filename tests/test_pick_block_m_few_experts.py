"""The row block that layers of fewer than 32 experts get."""
import pytest


@pytest.mark.parametrize("tokens,topk,experts,expected", [
    (128, 2, 8, 64),       # 32 rows per expert
    (132, 2, 8, 64),       # 33: one block of 64 still holds an expert
    (176, 2, 8, 64),       # 44
    (177, 2, 8, 128),      # 44.25: the busier experts would need a second block
    (352, 2, 16, 64),      # 44
    (256, 2, 17, 64),      # 30: twice the mean, as for any layer of fewer than 32 experts
    (280, 2, 17, 128),     # 33, but enough experts for loads to differ
    (238, 4, 28, 128),     # 34
    (400, 4, 32, 128),     # 50
])
def test_few_experts(tokens, topk, experts, expected):
    from pyhip_amd.fused_moe import pick_block_m
    assert pick_block_m(tokens, topk, experts) == expected


def test_bf16_activations_keep_their_rule():
    from pyhip_amd import _lib
    lib = _lib.load()
    assert [lib.pyhip_moe_pick_block_m(t, 2, 8, 4096, 1) for t in (16, 64, 128, 200, 4096)] == [16, 32, 64, 64, 64]
