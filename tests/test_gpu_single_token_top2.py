"""A single token of a top-2 layer: the down GEMM that also sums the slots, at the edges of what it serves."""
import pytest
import torch

import cases

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("H,I,splitk", [
    (512, 512, 0),          # four waves, a K-step for each
    (1024, 2560, 4),        # an uneven share of K-steps
    (512, 2048, 32),        # sixteen waves, a K-step for each
    (512, 16384, 0),        # sixteen waves, the largest rows that LDS takes
    (512, 16896, 0),        # one tile more: the two launches
    (2048, 2048, 16),       # a split that only the two launches have
    (512, 1024, 1),
])
def test_top2_token(H, I, splitk):
    from pyhip_amd import fused_moe
    L = cases.make_layer("", 1, seed=H + I, bias=True, E=4, k=2, H=H, I=I, router="softmax")
    w1, w1s, w2, w2s = cases.device_weights(L)
    b1, b2 = L.bias1.cuda() * 20, L.bias2.cuda() * 20
    hidden, tw = L.hidden.cuda(), torch.from_numpy(L.topk_w).cuda()
    print(f"top-2 token H={L.H} I={I} splitk={splitk}", flush=True)
    for drop in (None, 0, 1, 2):
        ids = L.topk_ids.copy()
        if drop is not None:
            ids[0, drop if drop < 2 else slice(None)] = -1
        ti = torch.from_numpy(ids).cuda()
        for dt in (torch.bfloat16, torch.float32):
            kw = dict(w1_scale=w1s, w2_scale=w2s, bias1=b1, bias2=b2, method="w4a16", splitk=splitk, dtype=dt)
            want = fused_moe(hidden, w1, w2, tw, ti, return_parts=True, **kw)[0]
            got = fused_moe(hidden, w1, w2, tw, ti, **kw)
            torch.cuda.synchronize()
            assert torch.equal(got, want) and (drop != 2 or (got == 0).all())
