"""The unique count of a training backprop is written to pinned memory by its
kernels; when a launch behind them fails, that write must not be left for the
thread's next dedup (tests/cpp/pending_head_check.cpp: the host code over a
pretended device)."""
import os
import subprocess

ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))
CSRC = os.path.join(ROOT, "nv-embedding-cache_amd", "csrc")


def test_no_write_to_the_head_is_left_behind(tmp_path):
    exe = str(tmp_path / "pending_head_check")
    src = [os.path.join(ROOT, "tests", "cpp", "pending_head_check.cpp")] + \
          [os.path.join(CSRC, f) for f in ("backprop.cpp", "dedup.cpp")]
    subprocess.run(["g++", "-O1", "-std=c++17", "-D__HIP_PLATFORM_AMD__", "-I/opt/rocm/include", "-I" + CSRC,
                    "-I" + os.path.join(ROOT, "include"), "-o", exe] + src, check=True, timeout=300)
    p = subprocess.run([exe], capture_output=True, text=True, timeout=60)
    assert p.returncode == 0 and "pending head ok" in p.stdout, p.stdout + p.stderr
