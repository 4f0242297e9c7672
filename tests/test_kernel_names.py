"""Names of gather kernels: what a plan reports is a kernel of the sources, and the benchmark finds that
kernel's counters by it."""
import os
import re

import bench
from backprojector_amd import roofline as rl

CSRC = os.path.join(os.path.dirname(os.path.dirname(os.path.abspath(__file__))), "backprojector_amd", "csrc")

# reported name -> the kernel's own (demangled) name
NAMES = {
    "confocal_lds_kernel_poly<CountRows, KZ=16, degree=2> (16x16x16 tiles, 8 pair parts)":
        "void bpx::confocal_lds_kernel_poly<bpx::(anonymous namespace)::CountRows, 16, 2, false>(bpx::LdsPolyArgs)",
    "confocal_lds_kernel_column<F32Rows, KZ=16, degree=3> (16x16x16 tiles, 1 pair part)":
        "void bpx::confocal_lds_kernel_column<bpx::(anonymous namespace)::F32Rows, 16, 3>(bpx::LdsPolyArgs)",
    "confocal_lds_kernel_column<Half16Rows<true>, KZ=8, degree=2> (16x16x8 tiles, 2 pair parts)":
        "void bpx::confocal_lds_kernel_column<bpx::(anonymous namespace)::Half16Rows<true>, 8, 2>(bpx::LdsPolyArgs)",
    "confocal_lds_kernel_column<ComplexRows, KZ=8, degree=2> (16x16x8 tiles, 2 pair parts)":
        "void bpx::confocal_lds_kernel_column<bpx::(anonymous namespace)::ComplexRows, 8, 2>(bpx::LdsPolyArgs)",
    "confocal_kernel_split<K=2> (8x8x8 tiles, 12 pair parts)":
        "void bpx::confocal_kernel_split<bpx::FusedSource<bpx::FusedF32>, 2, true, true>(bpx::ConfocalArgs, bpx::SplitPairs)",
    "paths_lds_kernel<grid> (16x16x8 tiles, 4 parts)": "void bpx::paths_lds_kernel<true, 8, false>(bpx::PathsLdsArgs)",
    "paths_lds_kernel<pairs> (16x16x8 tiles, 4 parts)": "void bpx::paths_lds_kernel<false, 8, false>(bpx::PathsLdsArgs)",
    "confocal_lds_kernel<KZ=8, waves=4> (16x16x8 tiles)":
        "void bpx::confocal_lds_kernel<bpx::FusedF32, 8, 4>(bpx::ConfocalArgs)",
}


def test_counters_are_found_by_the_reported_name():
    counts = {k: [{"SQ_INSTS_VALU": 1.0}] for k in NAMES.values()}
    for reported, kernel in NAMES.items():
        prefix = bench.device_kernel({"kernel": reported}, "f32", False)
        assert rl.find_signature(counts, prefix)[0] == kernel, (reported, prefix)


def test_reported_names_are_kernels():
    text = "".join(open(os.path.join(CSRC, f)).read() for f in sorted(os.listdir(CSRC)) if f.endswith(".hip"))
    kernels = set(re.findall(r"__global__[^;{]*?void (\w+)\(", text))
    api = open(os.path.join(CSRC, "bpx_api.cpp")).read()
    body = api[api.index("bpx_status bpx_plan_kernel_name("):api.index("bpx_status bpx_plan_benchmark(")]
    reported = set(re.findall(r'"(\w+_kernel\w*)', body))
    assert len(reported) >= 8 and reported <= kernels, reported - kernels
    assert all(r.split("<")[0] in reported for r in NAMES)
