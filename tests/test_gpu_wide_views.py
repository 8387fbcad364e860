"""bf16 activations at the true width of a padded layer, as columns of a very wide buffer: rows too far apart for 32-bit offsets are
widened first."""
import pytest
import torch

import cases

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("T,stride", [(64, 2 ** 24 - 8), (65, 2 ** 24 - 8), (3, 2 ** 24)])
def test_columns_of_a_wide_buffer(T, stride):
    from pyhip_amd import fused_moe
    L = cases.make_layer("", T, seed=T, E=8, k=1, H=960, I=512, router="softmax")
    w1, w1s, w2, w2s, _, _, hp, ip = cases.padded_device_weights(L)
    tw, ti = torch.from_numpy(L.topk_w).cuda(), torch.from_numpy(L.topk_ids).cuda()
    kw = dict(w1_scale=w1s, w2_scale=w2s, hidden_pad=hp, intermediate_pad=ip, method="w4a16", block_size_M=16)
    x = L.hidden.cuda()
    view = torch.empty_strided((T, L.H), (stride, 1), dtype=torch.bfloat16, device="cuda")
    view.copy_(x)
    print("columns of a wide buffer", T, stride, flush=True)
    assert hp == 64 and torch.equal(fused_moe(view, w1, w2, tw, ti, **kw), fused_moe(x, w1, w2, tw, ti, **kw))
