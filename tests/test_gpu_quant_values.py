"""The activation quantiser on every bf16 value."""
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


def test_infinities_and_nans_saturate_and_leave_their_block_alone():
    """A block with an infinity or a NaN has the scale byte of an infinity; the value itself becomes 6 of its own sign, and the
    finite values beside it what that scale makes of them."""
    from pyhip_amd.fused_moe import act_quant_mxfp4
    rng = np.random.default_rng(5)
    special = np.array([0x7F80, 0xFF80, 0x7FC0, 0xFFC0, 0x7F81, 0xFF81, 0x7FFF, 0xFFFF], np.uint32)
    bits = rng.permutation(np.arange(1 << 16, dtype=np.uint32)).reshape(128, 512)
    bits[(bits & 0x7F80) == 0x7F80] = 0x3F80
    bits[:, ::32] = rng.choice(special, (128, 16))
    at = (bits & 0x7F80) == 0x7F80
    print("quantiser values, infinities and NaNs", flush=True)
    q, s = act_quant_mxfp4(torch.from_numpy(bits.astype(np.uint16).view(np.int16)).view(torch.bfloat16).cuda())
    torch.cuda.synchronize()
    assert (cases.untranspose_act_scales(s.cpu().numpy(), 512) == 253).all()
    # the oracle's encoder at that scale (it has no rule for the infinities and NaNs themselves)
    finite = np.where(at, 0, bits)
    want = om.e2m1_encode_rne(np.ldexp((finite << 16).view(np.float32), 127 - 253))
    want[at] = np.where(bits[at] >> 15, 15, 7)
    codes = np.empty((128, 512), np.uint8)
    codes[:, 0::2], codes[:, 1::2] = q.cpu().numpy() & 15, q.cpu().numpy() >> 4
    assert (codes == want).all(), np.argwhere(codes != want)[:5]
