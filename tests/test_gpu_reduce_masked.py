"""The top-k reduction of large calls under an expert mask (two pieces of 16 bytes to a lane): rows that end inside the first piece,
inside the second and on the edges, more than eight slots, against sums in slot order."""
import pytest
import torch

from pyhip_amd import _lib

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("T,k,H", [(40000, 8, 8), (530, 8, 504), (520, 8, 512), (520, 8, 520), (270, 8, 1024), (260, 9, 1032), (150, 17, 1536),
                                   (90, 8, 2936)])
@pytest.mark.parametrize("f32", [False, True])
def test_masked_reduction(T, k, H, f32):
    assert T * k * H // 8 > 1 << 18                  # else the other kernel serves the call
    g = torch.Generator().manual_seed(T + H)
    E = 24
    x = torch.randn(T, k, H, generator=g).bfloat16()
    ids = torch.randint(-1, E + 1, (T, k), generator=g, dtype=torch.int32)
    mask = (torch.rand(E, generator=g) < 0.3).to(torch.int32)
    mask[:2] = torch.tensor([0, 1])
    kept = (ids >= 0) & (ids < E) & (mask[ids.clamp(0, E - 1).long()] != 0)
    want = torch.zeros(T, H)
    for s in range(k):
        want = torch.where(kept[:, s:s + 1], want + x[:, s].float(), want)
    out = torch.full((T, H), float("nan"), dtype=torch.float32 if f32 else torch.bfloat16, device="cuda")
    xd, idd, md = x.cuda(), ids.cuda(), mask.cuda()
    xd.view(T * k, H)[~kept.flatten().cuda()] = float("nan")
    local = torch.tensor([T - 3], dtype=torch.int32, device="cuda")
    print("masked reduction", T, k, H, f32, flush=True)
    lib = _lib.load()
    for n in (None, local):
        _lib.check(lib.pyhip_moe_topk_reduce_routed(xd.data_ptr(), out.data_ptr(), T, k, H, int(f32), idd.data_ptr(), E, md.data_ptr(),
                                                    None if n is None else n.data_ptr(), _lib.current_stream()))
        if n is not None:
            want[T - 3:] = 0
        assert torch.equal(out.cpu(), want.to(out.dtype))
