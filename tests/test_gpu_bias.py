"""Biases reach every tile height from wherever they lie: the MXFP4 GEMMs bring them to LDS four bytes at a time when the
tensor allows it and with ordinary loads when it is only element-aligned."""
import numpy as np
import pytest
import torch

import cases
from oracle import moe

pytestmark = pytest.mark.gpu


def _at_offset(t, elems):
    """the same values in a contiguous tensor that starts `elems` elements into its storage"""
    buf = torch.empty(t.numel() + elems, dtype=t.dtype, device=t.device)
    view = buf[elems:].view(t.shape)
    view.copy_(t)
    assert view.is_contiguous() and view.data_ptr() % 4 == 2 * elems % 4
    return view


@pytest.mark.parametrize("bm,T", [(16, 20), (32, 90), (64, 130), (128, 400), (160, 500), (192, 600), (256, 700), (288, 800)])
def test_biases_at_every_tile_height_and_alignment(bm, T):
    from pyhip_amd import fused_moe
    L = cases.make_layer("odd", T, seed=11, bias=True)
    w1, w1s, w2, w2s = cases.device_weights(L)
    # as large as the layer's own values: a bias of another channel, expert or tile is far outside the tolerance
    b1, b2 = L.bias1.cuda() * 100, L.bias2.cuda() * 100
    kw = dict(w1_scale=w1s, w2_scale=w2s, block_size_M=bm, dtype=torch.float32, method="a4w4")
    tw, ti = torch.from_numpy(L.topk_w).cuda(), torch.from_numpy(L.topk_ids).cuda()
    print(f"bias case bm={bm} T={T}", flush=True)
    outs = [fused_moe(L.hidden.cuda(), w1, w2, tw, ti, bias1=_at_offset(b1, o), bias2=_at_offset(b2, o), **kw) for o in (0, 1, 2)]
    torch.cuda.synchronize()
    assert torch.equal(outs[0], outs[1]) and torch.equal(outs[0], outs[2])
    f = lambda t: t.float().cpu().numpy()
    ref = moe.moe_ref(f(L.hidden), L.w1q, L.w1s, L.w2q, L.w2s, L.topk_w, L.topk_ids, act="a4", bias1=f(b1), bias2=f(b2))
    err = np.abs(f(outs[0]) - ref) / np.sqrt(np.mean(ref ** 2))
    print(f"beyond 1e-2 rms: {np.mean(err > 1e-2):.2e}, max {err.max():.2e}", flush=True)
    # as in the layer tests: bf16 roundings of the intermediate that go the other way may move a few elements by up to 0.1 rms
    assert np.mean(err > 1e-2) <= 2e-3 and err.max() <= 0.1
