"""Without a row block given, the options of the step-by-step path take the ladder's height, which they serve, also where the one-call
path's kernels have another."""
import pytest
import torch

import cases
from pyhip_amd import _lib

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("T,k,E,H,I", [
    (40, 2, 32, 512, 512),        # 16 rows and 32
    (1024, 2, 8, 1024, 512),      # 128 and 32
])
def test_options_keep_the_ladders_height(T, k, E, H, I):
    from pyhip_amd import fused_moe
    from pyhip_amd.fused_moe import pick_block_m
    rows = pick_block_m(T, k, E, H)
    assert rows in (16, 128) and _lib.load().pyhip_layer_block_m(T, k, E, E, H, I) == 32
    L = cases.make_layer("", T, seed=T, E=E, k=k, H=H, I=I, router="softmax")
    w1, w1s, w2, w2s = cases.device_weights(L)
    args = (L.hidden.cuda(), w1, w2, torch.from_numpy(L.topk_w).cuda(), torch.from_numpy(L.topk_ids).cuda())
    kw = dict(w1_scale=w1s, w2_scale=w2s, method="a4w4")
    want, parts = fused_moe(*args, return_parts=True, **kw)
    assert parts["block_m"] == rows and torch.equal(fused_moe(*args, **kw), want)
    assert torch.equal(fused_moe(*args, topk_reduce="last_arriver", **kw), want)
    # (two slots a token: 0 + a is exact and a + b is rounded to bf16 once here, there to float32 first)
    got = fused_moe(*args, topk_reduce="atomic", **kw)
    assert (got.float() - want.float()).norm() <= 2 ** -8 * want.float().norm()
