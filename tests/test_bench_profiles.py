"""The profiles that bench.py's line draws on are of the kernels its workloads
launch, and its GEMM figures leave out a product that the E-step took over."""
import json
import os

import bench
import cudamica_amd as ca

PROFILES = os.path.join(os.path.dirname(os.path.abspath(bench.__file__)), "profiles")


def test_profiles_are_of_the_kernels_that_run():
    seen = 0
    for f in sorted(os.listdir(PROFILES)):
        kind, _, rest = f.partition("_")
        if kind not in ("sq", "traffic") or not f.endswith(".json"):
            continue
        workload, _, prec = rest[:-5].rpartition("_")
        w = ca.WORKLOADS[workload]
        with open(os.path.join(PROFILES, f)) as fh:
            kernel = json.load(fh)["kernel"]
        assert kernel.startswith(bench.estep_kernel(w.n, w.M, w.m, bench.PRECISIONS[prec])), f
        seen += 1
    assert seen >= 4


def test_valu_rate_is_the_profiled_instructions_over_the_live_time():
    kernel = bench.estep_kernel(128, 4, 3, 16)
    v = bench.valu_rate("n128_T2M_M4", 16, kernel, 3.0)
    with open(os.path.join(PROFILES, "sq_n128_T2M_M4_bf16.json")) as fh:
        insts = json.load(fh)["counters"]["SQ_INSTS_VALU"]
    assert v["valu_insts_per_launch"] == insts
    assert abs(v["simd_cycles_per_inst"] - 1024 * 2.4e9 * 3.0e-3 / insts) < 1e-9
    assert bench.valu_rate("n128_T2M_M4", 16, "estep_kernel<3, false, 0>", 3.0) is None   # another kernel's


def test_estep_kernel_names():
    assert bench.estep_kernel(64, 1, 3, 32) == "estep_m1_unmix_kernel<3>"
    assert bench.estep_kernel(64, 1, 4, 32) == "estep_m1_kernel<4, true>"
    assert bench.estep_kernel(65, 1, 3, 16) == "estep_m1_kernel<3, false>"
    assert bench.estep_kernel(128, 4, 3, 32).startswith("estep_kernel<3, true, 0, false")
    assert bench.estep_kernel(600, 1, 2, 16).startswith("estep_kernel<2, false, 2, true")
