"""CPU checks of the host side of a layer call: pointers, and what the remembered sizes accept."""
import ctypes

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
