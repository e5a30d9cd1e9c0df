"""The scratch that ltx25_lora_add hands to its launches, on a CPU: tests/cpp/lora_scratch.cpp stands
in for the HIP runtime and the kernels' launchers and checks every launch against what the library
has allocated. One process per scenario, since the library's state lives as long as it does."""
import os
import shutil
import subprocess

import pytest

ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))
PKG = os.path.join(ROOT, "vpipe-ltx-2.5_amd")


@pytest.fixture(scope="module")
def exe(tmp_path_factory):
    hipcc = shutil.which("hipcc") or "/opt/rocm/bin/hipcc"
    if not os.path.exists(hipcc):
        pytest.skip("no hipcc")
    out = str(tmp_path_factory.mktemp("lora_scratch") / "lora_scratch")
    # host code only; its definitions come before the library's and the runtime's
    r = subprocess.run([hipcc, "-x", "hip", "--offload-host-only", "-std=c++17", "-O1", "-Wall",
                        "-I" + os.path.join(ROOT, "include"), "-I" + os.path.join(PKG, "csrc"),
                        os.path.join(ROOT, "tests", "cpp", "lora_scratch.cpp"), "-x", "none",
                        os.path.join(PKG, "libltx25_qlinear.so"), "-Wl,--export-dynamic", "-ldl",
                        "-Wl,-rpath," + PKG, "-o", out], capture_output=True, text=True)
    assert r.returncode == 0, r.stderr[-3000:]
    return out


def run(exe, *args):
    r = subprocess.run([exe, *map(str, args)], capture_output=True, text=True, timeout=60)
    assert r.returncode == 0, r.stdout + r.stderr


@pytest.mark.parametrize("rank", [96, 450, 1024])   # the y GEMM splits K at 1024, on 128 x 128 tiles
@pytest.mark.parametrize("before,after", [(0, 2), (2, 0)])   # AUTO, MID
def test_the_tile_switch_may_change_during_a_call(exe, rank, before, after):
    for n in range(1, 7):   # after the call's n-th plan
        run(exe, "tile_switch", rank, before, after, n)


# the plans under the fused route: r ahead of the y phase, both products on the dense GEMM; ranks
# and addresses of b that the kernels read as they are, and that need a copy
PLANS = [  # M, K, N, rank, bytes of b off 16-byte alignment
    (128, 4096, 1032, 32, 0), (128, 4096, 1032, 32, 2), (128, 4352, 1032, 12, 0),
    (33, 4096, 4104, 17, 0), (64, 1024, 1024, 450, 0), (100, 2048, 1000, 192, 6),
]


@pytest.mark.parametrize("M,K,N,rank,b_off", PLANS)
def test_streams_share_no_scratch(exe, M, K, N, rank, b_off):
    run(exe, "overlap", M, K, N, rank, b_off)


@pytest.mark.parametrize("M,K,N,rank,b_off", PLANS)
def test_a_call_prepares_its_capture(exe, M, K, N, rank, b_off):
    run(exe, "capture", M, K, N, rank, b_off)


def test_streams_that_come_and_go_keep_the_plans(exe):
    run(exe, "streams_come_and_go")


@pytest.mark.parametrize("M,K,N,rank", [(128, 4096, 1032, 32), (64, 1024, 1024, 450)])
def test_a_stream_handle_may_come_back(exe, M, K, N, rank):
    run(exe, "recycled_handle", M, K, N, rank)
