"""The activation quantiser on every finite bf16 value."""
import numpy as np
import pytest
import torch

import cases
from oracle import mxfp4 as om

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("order", ["by_magnitude", "mixed"])
def test_every_finite_bf16_value_matches_the_oracle(order):
    """By magnitude, a block's 32 values share one or two exponents, so every value meets the block scale it sets or nearly
    sets; mixed, most values are far below their block's scale."""
    from pyhip_amd.fused_moe import act_quant_mxfp4
    bits = np.arange(1 << 16, dtype=np.uint32)
    bits = bits[(bits & 0x7F80) != 0x7F80]                       # 65024 finite patterns, both zeros among them
    if order == "by_magnitude":
        bits = bits[np.argsort((bits & 0x7FFF) * 2 + (bits >> 15), kind="stable")]
    else:
        bits = np.random.default_rng(3).permutation(bits)
    bits = np.concatenate([bits, np.zeros(65536 - len(bits), np.uint32)])
    x = (bits << 16).view(np.float32).reshape(128, 512)
    print(f"quantiser values, {order}", flush=True)
    q, s = act_quant_mxfp4(torch.from_numpy(x).to(torch.bfloat16).cuda())
    torch.cuda.synchronize()
    oq, os_ = om.quantize_mxfp4(x)
    assert (cases.untranspose_act_scales(s.cpu().numpy(), 512) == os_).all()
    bad = np.argwhere(q.cpu().numpy() != oq)
    assert bad.size == 0, (len(bad), bad[:5])
