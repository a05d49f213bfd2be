"""What the library launches, without a GPU: its host code runs on a stand-in for the HIP runtime
(launch_trace.cpp) that writes every launch down, and the kernels' resources come from the built
library's own metadata."""
import os
import re
import shutil
import subprocess
import sys

import pytest
import yaml

from justgoal_amd import build
from justgoal_amd.geometry import DS_V3, QWEN3, ROUTING_SOFTMAX, Geometry

HERE = os.path.dirname(os.path.abspath(__file__))
LLVM = "/opt/rocm/llvm/bin"
CUS, LDS_PER_CU = 256, 160 * 1024
pytestmark = pytest.mark.skipif(not (shutil.which("g++") and os.path.exists(f"{LLVM}/llvm-readelf")),
                                reason="needs g++ and the ROCm toolchain")

# Calls moe_run_ex once per line of stdin: the eight geometry fields and T.
DRIVER = """
import ctypes, sys
ctypes.CDLL(sys.argv[1], ctypes.RTLD_GLOBAL)  # ahead of the runtime that the library is linked to
L = ctypes.CDLL(sys.argv[2])
P = ctypes.c_void_p
L.moe_run_ex.argtypes = [P] * 9 + [ctypes.c_int, ctypes.c_float, P, P, ctypes.c_int, P]
p = P(4096)
for line in sys.stdin:
    *g, T = map(int, line.split())
    print("#", flush=True)
    rc = L.moe_run_ex((ctypes.c_int * 8)(*g), p, p, p, p, p, p, p, p, 0, 1.0, p, p, T, None)
    assert rc == 0, (line, rc)
    ctypes.CDLL(None).fflush(None)
"""


def kernel_name(symbol):
    """Name and template arguments: "gemm2_wide_kernel<128,2,1>"."""
    name, args = re.search(r"\d([a-z][a-z0-9]*_[a-z0-9_]*kernel)(I(?:L[a-z]\d+E)+E)?", symbol).groups()
    return f"{name}<{','.join(re.findall('L[a-z]([0-9]+)E', args))}>" if args else name


@pytest.fixture(scope="module")
def plan(tmp_path_factory):
    """plan([(geometry, T), ...]) -> [[(kernel, grid, block), ...], ...]"""
    if not os.path.exists(build.LIB_PATH):
        build.build()
    trace = tmp_path_factory.mktemp("plan") / "trace.so"
    subprocess.run(["g++", "-O1", "-shared", "-fPIC", "-I/opt/rocm/include", "-o", str(trace),
                    os.path.join(HERE, "launch_trace.cpp")], check=True)

    def run(cases):
        lines = "".join(
            " ".join(map(str, (g.hidden, g.intermediate, g.num_experts, g.local_experts, g.top_k,
                               g.n_group, g.topk_group, g.routing_method, T))) + "\n"
            for g, T in cases)
        out = subprocess.run([sys.executable, "-c", DRIVER, str(trace), build.LIB_PATH], input=lines,
                             text=True, capture_output=True)
        assert out.returncode == 0, out.stderr
        calls = [c.strip().splitlines() for c in out.stdout.split("#")[1:]]
        assert len(calls) == len(cases)
        return [[(kernel_name(s), int(g), int(b)) for s, g, b in (x.split() for x in c)]
                for c in calls]

    return run


@pytest.fixture(scope="module")
def lds_bytes(tmp_path_factory):
    """{kernel: bytes of LDS that a workgroup takes}"""
    tmp = tmp_path_factory.mktemp("meta")
    lib = shutil.copy(build.LIB_PATH, tmp / "lib.so")
    subprocess.run([f"{LLVM}/llvm-objdump", "--offloading", str(lib)], check=True,
                   capture_output=True, cwd=tmp)
    out = {}
    for f in tmp.glob(f"lib.so.*{build.ARCH}"):
        notes = subprocess.run([f"{LLVM}/llvm-readelf", "--notes", str(f)], check=True,
                               capture_output=True, text=True).stdout
        meta = yaml.safe_load(re.search(r"---\n(.*?)\n\.\.\.", notes, re.S)[1])
        for k in meta.get("amdhsa.kernels", []):
            out[kernel_name(k[".name"])] = k[".group_segment_fixed_size"]
    return out


GEOMETRIES = [DS_V3, QWEN3] + [
    Geometry(H, I, E, El, 8, 1, 1, ROUTING_SOFTMAX)
    for H in (256, 384, 512, 640, 1024, 2048, 2560, 3072, 3584, 4096, 5120, 6144, 7680, 8192)
    for I in (128, 384, 1024, 1536) for E, El in ((64, 64), (128, 128), (256, 32), (256, 256))]


def test_persistent_grids_fit_the_chip(plan, lds_bytes):
    """A persistent GEMM's workgroups are all resident at once: one that had to wait for another to
    end would start over with empty rings."""
    cases = [(g, T) for g in GEOMETRIES
             for T in (1, 2, 5, 7, 12, 16, 33, 64, 128, 200, 512, 1024, 2048, 4096)]
    seen = set()
    for case, launches in zip(cases, plan(cases)):
        for kernel, grid, _ in launches:
            if kernel.startswith("gemm"):
                assert grid <= CUS * (LDS_PER_CU // lds_bytes[kernel]), (case, kernel, grid)
                seen.add(kernel)
    assert {f"gemm1_stream_kernel<1,{d},4>" for d in (4, 5, 6, 7, 8)} <= seen


def test_bench_names_the_kernels_that_run(plan):
    """bench.py names each GEMM's kernel by its own copy of the library's selection rules."""
    import bench
    from justgoal_amd import inputs as jin
    tokens = sorted({c.tokens for c in jin.CONFIGS.values()} | set(range(1, 40)) |
                    {t + d for t in (64, 95, 127, 128, 159, 160, 255, 256, 511, 512, 703, 704,
                                     1023, 1024, 2047, 2048) for d in (0, 1)})
    cases = [(g, T) for g in (DS_V3, QWEN3) for T in tokens]
    for (g, T), launches in zip(cases, plan(cases)):
        cfg = jin.Config("", g, T)
        names = [k.split("<")[0] for k, _, _ in launches if k.startswith("gemm")]
        assert names == [bench.gemm1_kernel_name(cfg), bench.gemm2_launch_name(cfg)], (g, T)


@pytest.mark.parametrize("geom,T,route,gemm2", [
    (DS_V3, 1, 1, 1), (DS_V3, 12, 1, 1), (DS_V3, 13, 2, 1), (DS_V3, 16, 2, 1), (DS_V3, 17, 2, 2),
    (QWEN3, 12, 1, 1), (QWEN3, 13, 1, 2), (QWEN3, 16, 1, 2), (QWEN3, 17, 2, 2)])
def test_few_token_calls_take_fewer_launches(plan, geom, T, route, gemm2):
    """Launches before GEMM1 (routing and permute) and after it (GEMM2 and combine)."""
    names = [k for k, _, _ in plan([(geom, T)])[0]]
    at = [i for i, k in enumerate(names) if k.startswith("gemm1")]
    assert len(at) == 1 and (at[0], len(names) - at[0] - 1) == (route, gemm2)
