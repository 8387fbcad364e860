"""The small stages around the GEMMs at the sizes where their split over waves has edges."""
import numpy as np
import pytest
import torch

from pyhip_amd import _lib

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("T,k,H", [(1, 1, 8), (3, 2, 504), (2, 8, 512), (5, 9, 520), (7, 4, 1032), (2, 33, 2880), (4001, 8, 256)])
@pytest.mark.parametrize("mode", ["plain", "ids", "mask", "local"])
@pytest.mark.parametrize("f32", [False, True])
def test_topk_reduce_edges(T, k, H, mode, f32):
    """Rows that are no whole number of 64-lane pieces, slots past one group of eight, dropped slots that hold NaN; against
    numpy's sums in slot order, which the kernel's single-precision additions must equal exactly."""
    g = torch.Generator().manual_seed(T * 100 + k)
    E = 16
    x = torch.randn(T, k, H, generator=g).to(torch.bfloat16)
    ids = torch.randint(0 if mode == "plain" else -1, E if mode == "plain" else E + 1, (T, k), generator=g, dtype=torch.int32)
    mask = (torch.arange(E) % 3 != 0).to(torch.int32) if mode == "mask" else None
    local = torch.tensor([T // 2], dtype=torch.int32) if mode == "local" else None
    keep = (ids >= 0) & (ids < E)
    if mask is not None:
        keep &= mask[ids.clamp(0, E - 1).long()] != 0
    if local is not None:
        keep &= (torch.arange(T) < T // 2)[:, None]
    x[~keep] = float("nan")
    ref = np.zeros((T, H), np.float32)
    xf = x.float().numpy()
    for s in range(k):
        ref += np.where(keep[:, s, None].numpy(), xf[:, s], np.float32(0))
    lib = _lib.load()
    P = _lib.dptr
    xd, idd = x.cuda(), ids.cuda()
    md, ld = (None if v is None else v.cuda() for v in (mask, local))
    out = torch.full((T, H), 7.0, dtype=torch.float32 if f32 else torch.bfloat16, device="cuda")
    print("topk_reduce", T, k, H, mode, f32, flush=True)
    if mode == "plain":
        _lib.check(lib.pyhip_moe_topk_reduce(P(xd), P(out), T, k, H, int(f32), None, _lib.current_stream()))
    else:
        _lib.check(lib.pyhip_moe_topk_reduce_routed(P(xd), P(out), T, k, H, int(f32), P(idd), E, P(md), P(ld),
                                                    _lib.current_stream()))
    want = torch.from_numpy(ref)
    assert torch.equal(out.cpu(), want if f32 else want.to(torch.bfloat16))
