"""The GEMMs' host-side routing on the CPU: tests/host_route/check.cpp, built
against libdgamd.so, looks at the lists that prepare_gemm makes of a batch
and at launch sizes, and tests/host_route/staged.cpp at the addresses of
csrc/staged.hpp, compiled for the host.  No GPU call is made."""
import os
import shutil
import subprocess

import pytest

ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))
PKG = os.path.join(ROOT, "distributed-gemm-thesis_amd")
ROCM = os.environ.get("ROCM_PATH", "/opt/rocm")

pytestmark = pytest.mark.skipif(shutil.which("g++") is None, reason="no host C++ compiler")


@pytest.fixture(scope="module")
def check(tmp_path_factory):
    exe = str(tmp_path_factory.mktemp("route") / "check")
    cmd = ["g++", "-O2", "-std=c++17", "-D__HIP_PLATFORM_AMD__", "-I" + os.path.join(ROOT, "include"),
           "-I" + os.path.join(PKG, "csrc"), "-I" + os.path.join(ROCM, "include"),
           os.path.join(ROOT, "tests", "host_route", "check.cpp"), "-o", exe, "-L" + PKG, "-ldgamd",
           "-L" + os.path.join(ROCM, "lib"), "-lamdhip64", "-Wl,-rpath," + PKG,
           "-Wl,-rpath," + os.path.join(ROCM, "lib")]
    b = subprocess.run(cmd, capture_output=True, text=True, timeout=300)
    assert b.returncode == 0, b.stderr[-3000:]

    def run(what, *args, **extra):
        env = {k: v for k, v in os.environ.items() if not k.startswith("DG_GEMM_")}
        r = subprocess.run([exe, what, *map(str, args)], capture_output=True, text=True, timeout=300, env=dict(env, **extra))
        assert r.returncode == 0, (r.stdout[-2000:], r.stderr[-3000:])
        assert what + ": ok" in r.stdout
        return r.stdout.split()
    return run


def test_tables_are_copied_once(check):
    """A batch of many segments costs the host one copy of its tables,
    whatever the number of tile choices that are compared."""
    check("bytes")


def test_parts_cover_each_problem_once(check):
    """Under every tile choice, cut or not: each element of each problem is
    in one part, each part's operands start at its rows and columns, the
    tile numbers of a list follow one another, and the kernels get only what
    they take."""
    check("parts")


def test_long_columns(check):
    """Leading dimensions of millions of elements: no problem that the
    direct-to-LDS kernels take goes to loads by elements instead, and only
    offsets that leave 32 bits do."""
    check("long")


def test_short_segments(check):
    """The choice between the kernels knows what a segment's end costs each:
    SUMMA in panels of 16 to 64 stays on the direct-to-LDS kernels."""
    check("short")


def test_short_fp32_products(check):
    """FP32 products of short K go to the kernel that is not slower than
    what they had before the register-staged tiles."""
    check("sgemm_short")


def test_first_use_times_distinct_choices(check):
    """An autotuned plan's first use times each distinct tile choice, and
    what is clearly slower only once."""
    check("trials")


def test_launch_dimensions(check):
    """The grids of the copies, the layer reduction and the generator stay
    below 2^32 threads a dimension at any size."""
    check("grids")


@pytest.mark.parametrize("value,choice", [(None, -1), ("direct", 0), ("128x128", 1), ("128x128whole", 2), ("64x64", 3),
                                          ("32x32", 4), ("256x128", -1), ("64", -1), ("", -1)])
def test_forced_choice(check, value, choice):
    """DG_GEMM_TILE: every choice by its name; anything else forces nothing,
    in FP64 and in FP32."""
    assert check("forced", **({} if value is None else {"DG_GEMM_TILE": value}))[0] == str(choice)


def test_staged_addresses(tmp_path):
    """Every element that the register-staged kernels load lies inside its
    operand and arrives at its own place, and 32-bit lane offsets are the
    true ones up to the longest leading dimension that takes them."""
    exe = str(tmp_path / "staged")
    hipcc = os.environ.get("HIPCC", os.path.join(ROCM, "bin", "hipcc"))
    b = subprocess.run([hipcc, "-x", "hip", "--offload-host-only", "-O1", "-std=c++17", "-I" + os.path.join(PKG, "csrc"),
                        os.path.join(ROOT, "tests", "host_route", "staged.cpp"), "-o", exe],
                       capture_output=True, text=True, timeout=300)
    assert b.returncode == 0, b.stderr[-3000:]
    r = subprocess.run([exe], capture_output=True, text=True, timeout=300)
    assert r.returncode == 0, (r.stdout[-2000:], r.stderr[-3000:])
    assert "staged: ok" in r.stdout


def test_forced_shapes_reach_their_kernels(check):
    """The FP64 shapes of the forced-kernel GPU test fall on the lists that
    they stand for under the direct choice."""
    from test_gpu_forced_kernels import EXPECT, SHAPES, geometry
    for oa, ob, m, n, k, off_a, off_b, kind in SHAPES:
        (_, _, lda), (_, _, ldb), _ = geometry(oa, ob, m, n, k, 2)
        x = [int(v) for v in check("lists", oa, ob, m, n, k, lda, ldb, off_a, off_b, DG_GEMM_TILE="direct")[:5]]
        assert EXPECT[kind](x[0], x[1], sum(x[2:])), (oa, ob, m, n, k, off_a, off_b, kind, x)
