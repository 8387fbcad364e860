"""What the kernels of pyhip_amd/co take as arguments: sizes as callers with a launcher of their own pack them.
A kernel whose struct grows reads past what such a caller gave it."""
import ctypes
import os
import struct

import pytest

from pyhip_amd import co_module as co

msgpack = pytest.importorskip("msgpack")


def _arguments(name):
    """kernel -> sizes of its arguments in order, from the metadata note that the compiler puts into a code object"""
    blob = open(os.path.join(co.CO_DIR, name + ".co"), "rb").read()
    at = blob.index(b"AMDGPU\0") - 12
    namesz, descsz, _ = struct.unpack_from("<III", blob, at)
    start = at + 12 + (namesz + 3) // 4 * 4
    meta = msgpack.unpackb(blob[start:start + descsz], strict_map_key=False)
    return {k[".name"]: [a[".size"] for a in k[".args"] if not a[".value_kind"].startswith("hidden")]
            for k in meta["amdhsa.kernels"]}


SORT, QUANT, ROUTE, W4A16 = 104, 56, 40, 152       # SortArgs, QuantArgs, RouteArgs, W4A16Args


def test_quantiser_struct():
    assert ctypes.sizeof(co.QuantArgs) == QUANT
    assert _arguments("moe_quant") == {"moe_act_quant_mxfp4_kernel": [QUANT]}


def test_sort_structs():
    got = _arguments("moe_sort")
    routed = {k: v for k, v in got.items() if "moe_sort_small_kernel" in k}
    assert len(routed) == 9 and all(v == [SORT, QUANT, ROUTE] for v in routed.values())
    assert got["moe_sort_hist_kernel"] == [SORT] and got["moe_sort_scatter_kernel"] == [SORT]
    assert got["moe_sort_scan_kernel"] == [SORT, QUANT]
    assert got["moe_sort_count_kernel"] == got["moe_sort_small_cols_kernel"] == got["moe_sort_scan_cols_kernel"] == [SORT, QUANT, 4]


def test_bf16_activation_struct():
    got = _arguments("moe_gemm_w4a16")
    assert sum("moe_gemm_w4a16_top2_kernel" in k for k in got) == 2 and len(got) == 17
    assert all(v == [W4A16] for v in got.values())


def test_mirrored_structs():
    reduce = _arguments("moe_reduce")
    for f32 in (0, 1):
        for routed in (0, 1):
            assert reduce[co.reduce_kernel_name(f32, routed)] == [8, 8, 8, 4, 4, 8, ctypes.sizeof(co.ReduceRouting)]
    gemm = _arguments("moe_gemm_mxfp4")
    assert gemm[co.gemm_kernel_name(2, 8)] == [ctypes.sizeof(co.GemmArgs)]
