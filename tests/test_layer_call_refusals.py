"""What the layer call refuses, and that it does so before it launches anything: the pointers here are no memory."""
import sys

import pytest
import torch

from pyhip_amd import _lib, fused_moe  # noqa: F401

pytestmark = pytest.mark.skipif(torch.cuda.is_available(), reason="no pointers like these where a launch could follow")


def _call(T, k, E, H, I, rows, w4a16, stride=None, cols=0, pad=0, gating=0, n_group=0, topk_group=0, inter_pad=0):
    lib, P = _lib.load(), 1 << 20
    ws = lib.pyhip_moe_forward_workspace_bytes(T, k, E, H, I, rows, w4a16)
    block = sys.modules["pyhip_amd.fused_moe"]._LAYER_CALL.pack(P, P, P, P, P, 0, 0, gating, P, P, 0, 0, P, P, H if stride is None else stride, ws, cols, 0,
                                                                T, k, E, H, I, pad, inter_pad, rows, w4a16, 0, 0, n_group, topk_group, 1, 7.0, E)
    return lib.pyhip_layer_forward(block, None)


@pytest.mark.parametrize("T", [1, 8, 200])
@pytest.mark.parametrize("w4a16", [0, 1])
def test_negative_group_counts(T, w4a16):
    """with and without a sort in front of the GEMMs"""
    with pytest.raises(RuntimeError, match="n_group=-1"):
        _lib.check(_call(T, 2, 64, 512, 512, 16, w4a16, gating=1 << 20, n_group=-1, topk_group=1), "layer")


@pytest.mark.parametrize("T,stride", [(64, 2 ** 24 - 8), (65, 2 ** 24 - 8), (64, 2 ** 24), (127, 2 ** 23 + 65536), (128, 2 ** 23), (1, 2 ** 24), (1, 960)])
def test_rows_at_the_true_width_are_asked_for_where_they_are_taken(T, stride):
    """bf16 activations of a padded layer: what the host is told about a row stride is what the call does with it"""
    sizes = (T, 1, 8, 1024, 512, 16, 1, 0)
    told = _lib.load().pyhip_layer_takes_cols(*sizes, stride)
    with pytest.raises(RuntimeError) as e:
        _lib.check(_call(T, 1, 8, 1024, 512, 16, 1, stride=stride, cols=960, pad=64), "layer")
    assert told == ("launch failed" in str(e.value)) != ("contiguous rows" in str(e.value))


@pytest.mark.parametrize("pad,inter_pad", [(-32, 0), (0, -512), (512, 0), (0, 1024), (544, 0), (0, 1056), (-512, -1024)])
@pytest.mark.parametrize("T", [3, 60])
def test_padding_outside_of_the_matrices(T, pad, inter_pad):
    """refused with MXFP4 activations; with bf16 ones taken by the kernels that look at no padding, as channels past an expert's matrix would be
    read and written by those that do"""
    assert _lib.load().pyhip_layer_takes_pairs(T, 2, 32, 512, 1024, 16, 0, 0) and _lib.load().pyhip_layer_takes_pairs(T, 2, 32, 512, 1024, 16, 1, 0)
    with pytest.raises(RuntimeError, match="hidden_pad=%d / inter_pad=%d" % (pad, inter_pad)):
        _lib.check(_call(T, 2, 32, 512, 1024, 16, 0, pad=pad, inter_pad=inter_pad), "layer")
    with pytest.raises(RuntimeError, match="moe_sort.* launch failed"):
        _lib.check(_call(T, 2, 32, 512, 1024, 16, 1, pad=pad, inter_pad=inter_pad), "layer")
