"""The fused kernels give the same words in whatever order a wave's lanes, and
a block's waves, run between two waits (CPU: compiled for the host and run lane
by lane, tests/cpp/lane_order_check.cpp)."""
import os
import subprocess

CPP = os.path.join(os.path.dirname(os.path.abspath(__file__)), "cpp")
CLANG = "/opt/rocm/llvm/bin/clang++"


def test_lane_order(tmp_path):
    exe = str(tmp_path / "lane_order_check")
    subprocess.check_call([CLANG, "-std=c++17", "-O0", "-march=x86-64-v3", "-ffp-contract=off", "-Wno-unknown-pragmas",
                           "-Wno-pass-failed", "-I", os.path.join(CPP, "host_hip"),
                           os.path.join(CPP, "lane_order_check.cpp"), "-lm", "-o", exe])
    r = subprocess.run([exe], capture_output=True, text=True, timeout=600)
    assert r.returncode == 0, r.stdout + r.stderr
