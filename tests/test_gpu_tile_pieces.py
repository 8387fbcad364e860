"""The tile list of the 128-row and taller tiles, dealt to the XCDs in one to eight pieces: every tile is worked on, whatever
the number of tiles.  The 64-row tile takes its list in runs: same layer, same bits."""
import pytest
import torch

import cases

pytestmark = pytest.mark.gpu


def _walk(ids, E, bm, width, columns, K):
    """(tiles, pieces, most tiles of a workgroup) of a GEMM whose weight tiles are `width` of `columns` columns; None: no schedule"""
    if K < (1536 if bm == 288 else 1024):
        return None
    count = torch.bincount(ids.flatten().cpu().long(), minlength=E)
    tiles = int(((count + bm - 1) // bm).sum()) * (columns // width)
    pieces = 1 if E < 32 or tiles < 1024 else 8 if tiles > 4096 else tiles // 512
    workgroups = torch.cuda.get_device_properties(0).multi_processor_count * (2 if bm <= 128 else 1)
    return tiles, pieces, -(-tiles // workgroups)


@pytest.mark.parametrize("name,T,bm,gate_up", [
    ("dsv3_s", 3000, 128, (856, 1)),       # a run for each XCD
    ("dsv3_s", 4500, 128, (1280, 2)),
    ("qwen3_s", 9000, 160, (1868, 3)),     # 32 experts, a busy one with a fifth of the rows
    ("dsv3_s", 13000, 192, (2304, 4)),
    ("dsv3_s", 18000, 128, (4620, 8)),     # a last piece that is short
    ("dsv3_s", 70000, 128, (17628, 8)),    # 35 tiles a workgroup
    ("mixtral_s", 9000, 128, (1160, 1)),   # few experts: runs
])
def test_every_tile_is_worked_on(name, T, bm, gate_up):
    from pyhip_amd import fused_moe
    L = cases.make_layer(name, 64, seed=5)
    w1, w1s, w2, w2s = cases.device_weights(L)
    g = torch.Generator().manual_seed(T)
    hidden = torch.randn(T, L.H, generator=g).to(torch.bfloat16).cuda()
    logits = torch.randn(T, L.E, generator=g) - (1.1 * torch.log(torch.arange(1.0, L.E + 1)) if name == "qwen3_s" else 0.0)
    tw, ti = torch.topk(torch.softmax(logits, -1), L.k, dim=-1)
    assert _walk(ti, L.E, bm, 128, L.I, L.H)[:2] == gate_up
    kw = dict(w1_scale=w1s, w2_scale=w2s, method="a4w4")
    print(f"tile pieces {name} T={T} bm={bm}", flush=True)
    got = fused_moe(hidden, w1, w2, tw.cuda(), ti.int().cuda(), block_size_M=bm, **kw)
    want = fused_moe(hidden, w1, w2, tw.cuda(), ti.int().cuda(), block_size_M=64, **kw)
    torch.cuda.synchronize()
    assert torch.equal(got, want)


# (a workgroup decodes its first 64 tiles at once; what comes after them is found one at a time, from a cursor that starts over
# when the walk comes back to the first piece)
@pytest.mark.parametrize("H,I,T,bm,gate_up,down", [
    (1536, 4096, 36000, 128, (8, True), (8, False)),
    (1536, 4096, 33000, 160, (8, True), (8, False)),
    (1536, 4096, 33000, 256, (8, True), (6, False)),
    (1536, 4096, 40000, 288, (8, True), (6, False)),     # this height reads the schedule from global memory
    (8192, 1536, 22000, 160, (8, False), (8, True)),
    (2048, 1024, 7500, 192, (2, False), (2, False)),
])
@pytest.mark.parametrize("router", ["softmax", "zipf"])
def test_every_tile_beyond_the_decoded_ones(H, I, T, bm, gate_up, down, router):
    from pyhip_amd import fused_moe, workloads
    shape = dict(E=40, k=4, H=H, I=I, router=router)
    W = workloads.make_weights(shape, "cuda", seed=3)
    hidden, tw, ti = workloads.make_inputs(shape, T, "cuda", seed=4)
    for K, (width, columns), (pieces, beyond) in ((H, (128, I), gate_up), (I, (256, H), down)):
        walk = _walk(ti, 40, bm, width, columns, K)
        assert walk[1] == pieces and (walk[2] > 64) == beyond, walk
    kw = dict(w1_scale=W["w1_scale"], w2_scale=W["w2_scale"], method="a4w4")
    print(f"tile pieces H={H} I={I} T={T} bm={bm} {router}", flush=True)
    got = fused_moe(hidden, W["w1"], W["w2"], tw, ti, block_size_M=bm, **kw)
    want = fused_moe(hidden, W["w1"], W["w2"], tw, ti, block_size_M=64, **kw)
    torch.cuda.synchronize()
    assert torch.equal(got, want)
