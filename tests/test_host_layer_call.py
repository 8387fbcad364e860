"""CPU checks of the host side of a layer call: pointers, and what the remembered sizes accept."""
import ctypes
import sys

import numpy as np
import pytest
import torch

from pyhip_amd import _lib, co_module


def test_pointers_keep_all_their_bits_outside_declared_argtypes():
    """a ``dptr`` among a code-object kernel's arguments, or given to a function whose argument types nobody declared,
    is a whole pointer (a plain integer would be cut to a 32-bit int there)"""
    x = torch.zeros(4)
    p = _lib.dptr(x)
    packed = co_module._as_c(p)
    assert ctypes.sizeof(packed) == 8 and packed.value == x.data_ptr()
    same = ctypes.CDLL(None).memchr             # memchr(p, 0, 1) returns p where *p is 0
    same.restype = ctypes.c_void_p
    assert same(p, 0, 1) == x.data_ptr()
    assert _lib.dptr(None) is None and _lib.addr(None) is None and _lib.addr(x) == x.data_ptr()


@pytest.mark.parametrize("method", ["a4w4", "w4a16", "auto"])
def test_row_block_of_any_integer_type(method):
    """a row block that converts to an integer is taken as one, and by its value at the time of the call"""
    import pyhip_amd.fused_moe  # noqa: F401
    plan = sys.modules["pyhip_amd.fused_moe"]._plan
    sizes = (300, 2, 8, 1024, 512, method)
    for bm in (16, 32, 64):
        want = plan(*sizes, bm)
        for v in (np.int64(bm), np.array(bm), torch.tensor(bm)):
            got = plan(*sizes, v)
            assert (got[0], int(got[1]), got[2]) == want
    t = torch.tensor(16)
    plan(*sizes, t)
    t.fill_(64)
    assert plan(*sizes, t)[2] == plan(*sizes, 64)[2]
    assert plan(300, np.array(2), *sizes[2:], 16) == plan(*sizes, 16)
    for v in (32.0, "32"):
        with pytest.raises((TypeError, ctypes.ArgumentError)):
            plan(*sizes, v)


@pytest.mark.parametrize("limit,want", [(None, 7.0), (0, 7.0), (3, 3.0), (0.1, np.float32(0.1)), (1e39, float("inf")), (sys.float_info.max, float("inf")),
                                        (float("inf"), float("inf")), (np.float32(2.5), 2.5), (torch.tensor(5.0), 5.0)])
def test_swiglu_limit_of_any_size(limit, want):
    """limits past float32 are taken, as infinity, also where the call goes over as one packed block"""
    import pyhip_amd.fused_moe  # noqa: F401
    m = sys.modules["pyhip_amd.fused_moe"]
    got = m._swiglu_limit(limit)
    assert got == want
    assert m._LAYER_CALL.unpack(m._LAYER_CALL.pack(*[0] * 32, got, 8))[-2] == want


def test_swiglu_limit_of_whatever_float_takes():
    import decimal
    import pyhip_amd.fused_moe  # noqa: F401
    limit = sys.modules["pyhip_amd.fused_moe"]._swiglu_limit
    assert limit("2.5") == limit(decimal.Decimal("2.5")) == limit(torch.tensor([2.5])) == 2.5
    with pytest.raises((TypeError, ValueError)):
        limit("none")
