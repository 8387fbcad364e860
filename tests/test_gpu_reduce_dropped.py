"""Slots that the routing drops cost the top-k reduction nothing, however the caller drops them."""
import pytest
import torch

from pyhip_amd import _lib

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("by", ["ids", "mask"])
def test_dropped_slots_are_not_read(by):
    """One slot in eight kept: with one written row for each token the call moves two ninths of what it moves with all
    eight kept, so it may not take more than 0.6 of the time (a kernel that reads every slot takes all of it; the inputs, 1 GiB
    in turn, do not fit the last-level cache)."""
    T, k, H, E = 4001, 8, 7168, 64
    lib, P = _lib.load(), _lib.dptr
    xs = [torch.randn(T, k, H, device="cuda", dtype=torch.bfloat16) for _ in range(3)]
    every = torch.arange(E, dtype=torch.int32).view(8, 8).repeat(T // 8 + 1, 1)[:T].contiguous()    # ids of one group of eight
    if by == "ids":
        few, mask = torch.where(torch.arange(k) == (torch.arange(T) % k)[:, None], every, -1), None
    else:
        few, mask = every, (torch.arange(E) % 8 == 0).to(torch.int32)
    out = torch.empty(T, H, dtype=torch.bfloat16, device="cuda")
    md = None if mask is None else mask.cuda()
    all_d, few_d = every.cuda(), few.contiguous().cuda()

    def call(x, ids, m):
        _lib.check(lib.pyhip_moe_topk_reduce_routed(P(x), P(out), T, k, H, 0, P(ids), E, P(m), None, _lib.current_stream()))

    def best(ids, m):
        times = []
        for _ in range(7):
            a, b = torch.cuda.Event(enable_timing=True), torch.cuda.Event(enable_timing=True)
            call(xs[0], ids, m)
            a.record()
            for i in range(12):
                call(xs[i % 3], ids, m)
            b.record()
            torch.cuda.synchronize()
            times.append(a.elapsed_time(b))
        return min(times)

    print("reduce with dropped slots", by, flush=True)
    whole, part = best(all_d, None), best(few_d, md)
    assert part < 0.6 * whole, (part, whole)
    call(xs[1], few_d, md)
    kept = few >= 0 if mask is None else mask[every.long()] != 0
    want = torch.where(kept[:64, :, None], xs[1][:64].cpu().float(), 0.0).sum(1).to(torch.bfloat16)    # one term each: exact
    assert torch.equal(out[:64].cpu(), want)
