"""ctypes binding of ``libpyhip_moe.so`` (the C ABI declared in ``include/pyhip_moe.h``).

There is no CPU fallback: if the library is missing, loading raises.
"""
import ctypes
import os

import torch

_HERE = os.path.dirname(os.path.abspath(__file__))
LIB_PATH = os.path.join(_HERE, "libpyhip_moe.so")

_current_device = torch.cuda.current_device
_raw_stream = getattr(torch._C, "_cuda_getCurrentRawStream", None)      # (a CPU-only torch has none)

_c = ctypes
_P, _I, _L, _F = _c.c_void_p, _c.c_int, _c.c_int64, _c.c_float

#: symbol -> (restype, argtypes); the single source the loader and the export test share
SIGNATURES = {
    "pyhip_moe_abi_version": (_I, []),
    "pyhip_moe_last_error": (_c.c_char_p, []),
    "pyhip_moe_topk_softmax": (_I, [_P, _I, _I, _I, _I, _P, _P, _P]),
    "pyhip_moe_topk_grouped_sigmoid": (_I, [_P, _I, _I, _I, _I, _I, _I, _P, _P, _P]),
    "pyhip_moe_sorting_max_blocks": (_L, [_L, _I, _I, _I]),
    "pyhip_moe_sorting_workspace_bytes": (_L, [_L, _I, _I]),
    "pyhip_moe_schedule_words": (_L, [_I]),
    "pyhip_moe_sorting": (_I, [_P, _P, _I, _I, _I, _I, _P, _P, _P, _P, _P, _P, _P, _P, _L, _P, _L, _P]),
    "pyhip_moe_pick_block_m": (_I, [_L, _I, _I, _I, _I]),
    "pyhip_moe_pick_w4a16": (_I, [_L, _I, _I, _I]),
    "pyhip_moe_zero_fill": (_I, [_P, _L, _P]),
    "pyhip_moe_forward_workspace_bytes": (_L, [_L, _I, _I, _I, _I, _I, _I]),
    "pyhip_moe_forward": (_I, [_P, _L, _P, _P, _P, _P, _P, _P, _P, _P, _P, _P, _P, _I, _I, _I, _I, _I, _I, _I, _I, _I, _I, _I,
                               _I, _F, _P, _L, _P]),
    "pyhip_moe_forward_cols": (_I, [_P, _L, _I, _P, _P, _P, _P, _P, _P, _P, _P, _P, _P, _P] + [_I] * 12 + [_F, _P, _L, _P]),
    "pyhip_moe_route_sorting": (_I, [_P, _I, _I, _I, _I, _I, _I, _I, _P, _P, _P, _P, _P, _P, _P, _P, _P, _P, _L, _P, _L, _L, _I,
                                     _P, _P, _P]),
    "pyhip_moe_forward_routed": (_I, [_P, _L, _P, _P, _P, _P, _P, _P, _P, _I, _I, _I, _P, _P, _P, _P, _P, _I, _I, _I, _I,
                                      _I, _I, _I, _I, _I, _I, _I, _I, _F, _P, _L, _P]),
    "pyhip_moe_forward_static_capacity": (_L, []),
    "pyhip_moe_forward_static": (_I, [_P, _L, _P, _P, _P, _P, _P, _P, _P, _P, _P, _P, _P, _I, _I, _I, _I, _I, _I, _I, _I, _I, _I, _I,
                                      _I, _F, _P]),
    "pyhip_moe_sorting_quant": (_I, [_P, _P, _I, _I, _I, _I, _P, _P, _P, _P, _P, _P, _P, _P, _L, _P, _L, _L, _I, _P, _P, _P]),
    "pyhip_moe_act_scale_stride": (_L, [_I]),
    "pyhip_moe_act_quant_mxfp4": (_I, [_P, _L, _L, _I, _P, _P, _P, _P]),
    "pyhip_moe_gemm1_mxfp4": (_I, [_P, _P, _P, _P, _P, _P, _P, _P, _P, _P, _P, _P, _I, _I, _I, _I, _I, _I, _I, _I, _L, _I, _F, _P]),
    "pyhip_moe_gemm2_mxfp4": (_I, [_P, _P, _P, _P, _P, _P, _P, _P, _P, _P, _P, _I, _I, _I, _I, _I, _I, _I, _I, _L, _P]),
    "pyhip_moe_gemm1_mxfp4_lds": (_I, [_P, _P, _P, _P, _P, _P, _P, _P, _P, _P, _P, _P, _I, _I, _I, _I, _I, _L, _I, _F, _P]),
    "pyhip_moe_gemm2_mxfp4_lds": (_I, [_P, _P, _P, _P, _P, _P, _P, _P, _P, _P, _P, _I, _I, _I, _I, _I, _L, _P]),
    "pyhip_moe_gemm2_mxfp4_atomic": (_I, [_P, _P, _P, _P, _P, _P, _P, _P, _P, _P, _P, _I, _I, _I, _I, _I, _I, _L, _P]),
    "pyhip_moe_gemm2_mxfp4_reduce": (_I, [_P, _P, _P, _P, _P, _P, _P, _P, _P, _P, _P, _P, _P, _P, _P, _P, _I,
                                          _I, _I, _I, _I, _I, _I, _L, _P]),
    "pyhip_moe_gemm1_w4a16": (_I, [_P, _P, _P, _P, _P, _P, _P, _P, _I, _I, _I, _I, _I, _I, _L, _I, _I, _F, _P]),
    "pyhip_moe_gemm2_w4a16": (_I, [_P, _P, _P, _P, _P, _P, _P, _P, _P, _I, _I, _I, _I, _I, _I, _L, _I, _P]),
    "pyhip_moe_gemm1_w4a16_token": (_I, [_P, _P, _P, _P, _P, _P, _P, _P, _I, _I, _I, _I, _I, _I, _F, _P]),
    "pyhip_moe_gemm2_w4a16_token": (_I, [_P, _P, _P, _P, _P, _P, _P, _P, _P, _I, _I, _I, _I, _I, _P]),
    "pyhip_moe_probe_mfma_stream": (_I, [_I, _I, _P, _L, _P, _I, _P, _P]),
    "pyhip_moe_topk_reduce": (_I, [_P, _P, _L, _I, _I, _I, _P, _P]),
    "pyhip_moe_topk_reduce_routed": (_I, [_P, _P, _L, _I, _I, _I, _P, _I, _P, _P, _P]),
}

#: what fused_moe.py calls and the header does not declare: the layer call as one block of arguments, and its choices
INTERNAL = {
    "pyhip_layer_forward": (_I, [_c.c_char_p, _P]),
    "pyhip_layer_block_m": (_I, [_L, _I, _I, _I, _I, _I]),
    "pyhip_layer_takes_pairs": (_I, [_L, _I, _I, _I, _I, _I, _I, _I]),
    "pyhip_layer_sums": (_I, [_L, _I, _I, _I, _I, _I]),
    "pyhip_layer_takes_cols": (_I, [_L, _I, _I, _I, _I, _I, _I, _I, _L]),
}

_lib = None


class PyhipError(RuntimeError):
    pass


def load():
    global _lib
    if _lib is None:
        if not os.path.exists(LIB_PATH):
            raise PyhipError(
                "%s is missing: build it with `python -m pyhip_amd.build` (needs hipcc); "
                "there is no fallback path" % LIB_PATH)
        lib = ctypes.CDLL(LIB_PATH)
        for name, (res, args) in [*SIGNATURES.items(), *INTERNAL.items()]:
            fn = getattr(lib, name)
            fn.restype, fn.argtypes = res, args
        _lib = lib
    return _lib


def check(rc, what=""):
    if rc != 0:
        msg = load().pyhip_moe_last_error().decode("utf-8", "replace")
        raise PyhipError("%s failed (code %d): %s" % (what or "pyhip_moe call", rc, msg))


def addr(t):
    """device address of a torch tensor (or None) as a plain integer, the cheapest form of a pointer: only for functions
    whose ``argtypes`` say ``c_void_p``, as those of ``load()`` do (ctypes cuts an integer to 32 bits without them)"""
    return None if t is None else t.data_ptr()


def address(t):
    """the same for a packed block of arguments, where None is 0"""
    return 0 if t is None else t.data_ptr()


def stream_handle():
    """the current torch stream's handle as an integer, without the Stream object that ``torch.cuda.current_stream()``
    builds; for the same functions as ``addr``"""
    return _raw_stream(_current_device())


def dptr(t):
    """device pointer of a torch tensor (or None) as a ``c_void_p``: also right for functions without ``argtypes`` and
    among the arguments of a ``co_module.Kernel``, where an integer is a 32-bit int"""
    return None if t is None else ctypes.c_void_p(t.data_ptr())


def current_stream():
    """``stream_handle()`` as a ``c_void_p``"""
    return ctypes.c_void_p(stream_handle())
