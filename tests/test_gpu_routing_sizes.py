"""Router and sort on both sides of the number of tokens from which the router has a launch of its own."""
import pytest
import torch

from pyhip_amd import routing

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("T", [1, 7, 8, 63])
@pytest.mark.parametrize("E,grouped", [(64, False), (256, True), (512, False)])
def test_routed_call_equals_its_steps(T, E, grouped):
    import cases
    from pyhip_amd import fused_moe, fused_moe_routed
    L = cases.make_layer("dsv3_s", T, seed=9, E=E, k=8, H=512, I=512, router="softmax")
    logits = torch.randn(T, E, generator=torch.Generator().manual_seed(T + E)).cuda()
    w1, w1s, w2, w2s = cases.device_weights(L)
    kw = dict(num_expert_group=8, topk_group=4) if grouped else {}
    w, ids = routing.grouped_topk(logits, 8, True, 8, 4) if grouped else routing.fused_topk(None, logits, 8, True)
    print(f"routed sizes T={T} E={E} grouped={grouped}", flush=True)
    for nloc in (None, max(T - 3, 0)):
        n = None if nloc is None else torch.tensor([nloc], dtype=torch.int32, device="cuda")
        ref = fused_moe(L.hidden.cuda(), w1, w2, w, ids, w1_scale=w1s, w2_scale=w2s, num_local_tokens=n)
        out, tw, ti = fused_moe_routed(L.hidden.cuda(), w1, w2, logits, 8, True, w1_scale=w1s, w2_scale=w2s, num_local_tokens=n,
                                       return_routing=True, **kw)
        torch.cuda.synchronize()
        assert torch.equal(ti, ids) and torch.equal(tw, w) and torch.equal(out, ref)
