"""The tile height of a layer call whose sizes are known: a served one for any sizes, the ladder's where no other is clearly better."""
import random

import pytest

from pyhip_amd import _lib


@pytest.mark.parametrize("tokens,topk,experts,local,hidden,inter,want", [
    (493, 2, 8, 8, 1024, 512, 16),           # few tiles: the ladder has 160 rows
    (1024, 2, 8, 8, 1024, 512, 32),          # 128
    (446, 1, 8, 8, 2560, 2048, 32),          # 128
    # where the ladder stays
    (4096, 2, 8, 8, 4096, 14336, 128), (4096, 4, 128, 128, 3072, 3072, 160), (2048, 8, 128, 128, 4096, 1536, 160),
    (4001, 8, 256, 32, 7168, 2048, 160), (8192, 8, 256, 256, 7168, 2048, 288), (128, 8, 256, 256, 7168, 2048, 32),
    (16, 4, 128, 128, 3072, 3072, 16), (64, 2, 8, 8, 1024, 512, 32),
    # two rows per expert and more, in 32 experts and more: 32 rows (the ladder: 16)
    (80, 8, 256, 256, 7168, 2048, 32), (63, 8, 256, 256, 7168, 2048, 16), (17, 4, 32, 32, 4096, 4096, 32), (16, 4, 32, 32, 4096, 4096, 16),
    (20, 4, 31, 31, 4096, 4096, 16),
    # five and more, hidden 3072 and more: 64 (32)
    (300, 8, 256, 256, 7168, 2048, 64), (160, 4, 128, 128, 3072, 3072, 64), (159, 4, 128, 128, 3072, 3072, 32), (150, 4, 60, 60, 2048, 1536, 32),
])
def test_known_choices(tokens, topk, experts, local, hidden, inter, want):
    assert _lib.load().pyhip_layer_block_m(tokens, topk, experts, local, hidden, inter) == want


def test_any_sizes_get_a_served_height():
    lib, rng = _lib.load(), random.Random(0)
    served = {16, 32, 64, 128, 160, 192, 256, 288}
    for _ in range(3000):
        experts = rng.choice([1, 2, 3, 8, 60, 256, 2048, 5000])
        a = (int(2 ** rng.uniform(0, 23)), rng.randint(1, 255), experts, rng.randint(1, experts), rng.randrange(512, 16897, 512),
             rng.randrange(512, 16897, 512))
        assert lib.pyhip_layer_block_m(*a) in served, a
    for a in ((0, 2, 8, 8, 1024, 512), (64, 0, 8, 8, 1024, 512), (64, 2, 8, 0, 1024, 512)):
        assert lib.pyhip_layer_block_m(*a) == lib.pyhip_moe_pick_block_m(a[0], a[1], a[2], a[4], 0)


@pytest.mark.parametrize("tokens,topk,experts,local,hidden,inter,want", [
    # fewer tiles than CUs, but a long K loop and more lower tiles than run at once: measured slower by 12 to 40 %
    (216, 2, 8, 8, 7168, 3072, 128), (377, 2, 12, 12, 4096, 2048, 128), (348, 2, 8, 8, 4608, 2560, 128), (466, 2, 8, 8, 6144, 2560, 160),
    (193, 2, 8, 8, 4608, 3072, 128), (1153, 2, 24, 24, 5120, 512, 128), (1016, 2, 8, 8, 2560, 1024, 128),
    # few enough of them
    (371, 1, 8, 8, 6656, 512, 32),
    # the few-token kernels serve the ladder's height: the estimate is not of them
    (83, 2, 8, 8, 1536, 3584, 64), (135, 1, 8, 8, 4096, 1536, 64), (324, 1, 16, 16, 2048, 1024, 64),
])
def test_lower_tiles_only_where_they_cannot_lose_much(tokens, topk, experts, local, hidden, inter, want):
    assert _lib.load().pyhip_layer_block_m(tokens, topk, experts, local, hidden, inter) == want


@pytest.mark.parametrize("tokens,topk,experts,hidden,inter,rows,w4a16,want", [
    # a GEMM of 512 columns, more workgroups than few follow one another on a CU: measured slower by 2 to 20 % with MXFP4 activations
    (192, 8, 384, 512, 512, 16, 0, 0), (106, 8, 384, 512, 1536, 16, 0, 0), (107, 6, 160, 512, 512, 32, 0, 0), (80, 8, 128, 1024, 512, 32, 0, 0),
    (96, 8, 512, 4096, 512, 16, 0, 0), (96, 8, 256, 2048, 512, 64, 0, 0),
    (253, 6, 160, 1024, 1024, 64, 0, 0),
    # few of them, no sort, 16-row blocks of the middle sizes, or 1024 columns
    (253, 6, 160, 1024, 1024, 32, 0, 1), (60, 4, 32, 1024, 1024, 64, 0, 1),
    (11, 6, 160, 512, 512, 16, 0, 1), (8, 8, 384, 512, 512, 16, 0, 1), (96, 8, 256, 2048, 512, 16, 0, 1), (16, 4, 8, 512, 512, 32, 0, 1),
    (192, 8, 384, 1024, 1024, 32, 0, 1), (192, 8, 512, 3072, 1024, 32, 0, 1),
    # bf16 activations: only blocks that pass through LDS
    (253, 6, 160, 512, 1024, 16, 1, 0), (160, 6, 160, 512, 1024, 16, 1, 1), (253, 6, 160, 1024, 512, 16, 1, 1),
])
def test_few_token_kernels_only_where_their_k_loop_is_long_enough(tokens, topk, experts, hidden, inter, rows, w4a16, want):
    assert _lib.load().pyhip_layer_takes_pairs(tokens, topk, experts, hidden, inter, rows, w4a16, 0) == want


@pytest.mark.parametrize("tokens,topk,experts,hidden,inter,want", [
    # where they do not serve the higher block the ladder's height stays
    (192, 8, 512, 512, 512, 16), (96, 8, 256, 2048, 512, 16), (320, 8, 512, 4096, 512, 32),
    # 64 rows not with 1024 columns in the down GEMM
    (512, 8, 512, 3072, 1024, 32), (180, 8, 128, 4096, 1536, 64),
])
def test_higher_blocks_only_where_the_few_token_kernels_serve_them(tokens, topk, experts, hidden, inter, want):
    assert _lib.load().pyhip_layer_block_m(tokens, topk, experts, experts, hidden, inter) == want


@pytest.mark.parametrize("tokens,topk,experts,hidden,inter,rows,want", [
    # a handful of experts: the persistent kernels' tiles make most of one round of the chip
    (322, 2, 28, 7168, 1024, 64, 0), (322, 2, 28, 4096, 1024, 64, 0), (92, 4, 24, 7168, 1024, 64, 0), (96, 4, 24, 5120, 1024, 32, 0),
    # too few of them, as many as an uneven router takes into a second round, or few rows
    (92, 2, 8, 7168, 2048, 64, 1), (230, 2, 20, 5120, 1536, 64, 1), (190, 2, 20, 4096, 2048, 64, 1), (76, 2, 8, 4096, 2048, 64, 1), (140, 2, 28, 7168, 1024, 32, 1),
    (280, 2, 28, 4096, 1024, 64, 1), (322, 2, 28, 2048, 1024, 64, 1),
    # with or without a sort
    (64, 2, 8, 7168, 1536, 32, 1), (64, 2, 8, 1024, 512, 32, 1), (64, 2, 8, 7168, 1536, 16, 0),
])
def test_few_token_kernels_against_full_rounds_of_tiles(tokens, topk, experts, hidden, inter, rows, want):
    assert _lib.load().pyhip_layer_takes_pairs(tokens, topk, experts, hidden, inter, rows, 0, 0) == want


@pytest.mark.parametrize("tokens,topk,experts,held,hidden,inter,want", [
    (1, 8, 64, 64, 1536, 1536, 1), (1, 4, 64, 64, 3072, 3072, 1), (1, 8, 64, 64, 7168, 2048, 1), (1, 1, 64, 64, 512, 4096, 1), (1, 8, 16, 16, 1024, 2048, 1),
    (2, 8, 128, 128, 4096, 4096, 1), (1, 8, 32, 4, 4096, 4096, 1),
    # a token's slots one after the other take longer than the reduction does: up to 31 % more of the layer call than before these kernels
    (1, 8, 60, 60, 1536, 3584, 0), (1, 8, 64, 64, 2048, 2048, 0), (1, 4, 64, 64, 2048, 4096, 0), (2, 6, 96, 96, 1024, 3072, 0), (1, 8, 32, 32, 4096, 4096, 0),
])
def test_slots_are_summed_in_the_down_gemm_only_where_they_are_short(tokens, topk, experts, held, hidden, inter, want):
    assert _lib.load().pyhip_layer_sums(tokens, topk, experts, held, hidden, inter) == want


@pytest.mark.parametrize("tokens,topk,experts,local,hidden,inter,want", [
    # the ladder's height leaves nearly half of the CUs without a tile: 20 to 35 % less with lower ones
    (930, 1, 28, 28, 5120, 512, 32), (419, 2, 8, 8, 6144, 1024, 64), (289, 2, 8, 8, 5120, 1024, 32), (1130, 1, 8, 8, 6656, 1536, 64), (710, 1, 8, 8, 6656, 1024, 64),
    # more tiles than that
    (484, 1, 8, 8, 6656, 3584, 128), (200, 2, 8, 8, 6656, 3072, 128), (1009, 8, 128, 16, 4096, 1536, 128),
])
def test_lower_tiles_where_the_ladder_leaves_half_of_the_chip(tokens, topk, experts, local, hidden, inter, want):
    assert _lib.load().pyhip_layer_block_m(tokens, topk, experts, local, hidden, inter) == want
