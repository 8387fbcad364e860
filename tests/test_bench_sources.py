"""The digests beside the benchmark's traffic counters cover every file that the counted kernels are compiled from."""
import importlib.util
import os
import re

ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))
CSRC = os.path.join(ROOT, "pyhip_amd", "csrc")


def test_digests_cover_the_kernels_includes():
    spec = importlib.util.spec_from_file_location("bench", os.path.join(ROOT, "bench.py"))
    bench = importlib.util.module_from_spec(spec)
    spec.loader.exec_module(bench)
    kernels = set()
    for line, names in bench.KERNEL_SOURCES.items():
        for name in names:
            for inc in re.findall(r'^#include "(.+?)"', open(os.path.join(CSRC, name)).read(), re.M):
                assert inc in names, (line, name, inc)
        kernels.update(n for n in names if n.endswith(".hip"))
        assert re.fullmatch("[0-9a-f]{64}", bench.kernel_sources_digest(line))
    assert kernels == {"moe_gemm_mxfp4.hip", "moe_gemm_pairs.hip"}
