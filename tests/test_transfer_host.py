"""Worker threads of the memory manager, large host copies and the capture of
launches on the host (no GPU): the sources are built with host stand-ins for
the HIP calls they make, and C++ drivers check them."""
import os
import shutil
import subprocess

import pytest

ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))
HERE = os.path.join(ROOT, "tests", "memman_host")
CSRC = os.path.join(ROOT, "imagevis3d_amd", "csrc")


def run(tmp_path, *sources, flags=("-fsanitize=address,undefined",)):
    exe = str(tmp_path / "host_test")
    cmd = ["g++", "-std=c++17", "-O1", "-g", *flags, "-D__HIP_PLATFORM_AMD__", "-I/opt/rocm/include",
           *sources, os.path.join(HERE, "hip_stub.cpp"), "-lpthread", "-o", exe]
    subprocess.run(cmd, check=True, capture_output=True, text=True)
    r = subprocess.run([exe], capture_output=True, text=True, timeout=120,
                       env={**os.environ, "ASAN_OPTIONS": "detect_leaks=0"})
    print(r.stdout, r.stderr)
    assert r.returncode == 0 and "ALL OK" in r.stdout, r.stdout + r.stderr


pytestmark = pytest.mark.skipif(shutil.which("g++") is None or not os.path.isdir("/opt/rocm/include"),
                                reason="needs g++ and the ROCm headers")


def test_workers(tmp_path):
    run(tmp_path, os.path.join(HERE, "workers_test.cpp"), os.path.join(CSRC, "memman.cpp"))


def test_large_copies(tmp_path):
    run(tmp_path, os.path.join(HERE, "transfer_test.cpp"), os.path.join(HERE, "transfer_stub.cpp"),
        os.path.join(CSRC, "transfer.cpp"), os.path.join(CSRC, "memman.cpp"))


def test_one_graph_per_kernel_variant(tmp_path):
    run(tmp_path, os.path.join(HERE, "graph_test.cpp"), os.path.join(HERE, "transfer_stub.cpp"),
        os.path.join(CSRC, "renderer.cpp"), os.path.join(CSRC, "memman.cpp"),
        flags=("-Wl,--unresolved-symbols=ignore-all",))
