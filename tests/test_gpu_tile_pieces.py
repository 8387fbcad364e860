"""The tile list of the 128-row and taller tiles, dealt to the XCDs in one to eight pieces: every tile is worked on, whatever
the number of tiles.  The 64-row tile takes its list in runs: same layer, same bits."""
import pytest
import torch

import cases

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("name,T,bm", [
    ("dsv3_s", 3000, 128),       # about 900 down tiles of 128 rows: runs
    ("dsv3_s", 4500, 128),       # 1300: two pieces
    ("qwen3_s", 9000, 160),      # 32 experts, a busy one with a fifth of the rows
    ("dsv3_s", 13000, 192),      # 1900: three
    ("dsv3_s", 18000, 128),      # 4700: eight, a last piece that is short
    ("dsv3_s", 70000, 128),      # more than 64 tiles a workgroup: beyond the decoded table
    ("mixtral_s", 9000, 128),    # few experts: runs
])
def test_every_tile_is_worked_on(name, T, bm):
    from pyhip_amd import fused_moe
    L = cases.make_layer(name, 64, seed=5)
    w1, w1s, w2, w2s = cases.device_weights(L)
    g = torch.Generator().manual_seed(T)
    hidden = torch.randn(T, L.H, generator=g).to(torch.bfloat16).cuda()
    logits = torch.randn(T, L.E, generator=g) - (1.1 * torch.log(torch.arange(1.0, L.E + 1)) if name == "qwen3_s" else 0.0)
    tw, ti = torch.topk(torch.softmax(logits, -1), L.k, dim=-1)
    kw = dict(w1_scale=w1s, w2_scale=w2s, method="a4w4")
    print(f"tile pieces {name} T={T} bm={bm}", flush=True)
    got = fused_moe(hidden, w1, w2, tw.cuda(), ti.int().cuda(), block_size_M=bm, **kw)
    want = fused_moe(hidden, w1, w2, tw.cuda(), ti.int().cuda(), block_size_M=64, **kw)
    torch.cuda.synchronize()
    assert torch.equal(got, want)
