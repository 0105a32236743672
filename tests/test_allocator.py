"""The caching allocator over stubbed device memory, in a program of its own (no GPU)."""
import os
import subprocess

HERE = os.path.dirname(os.path.abspath(__file__))
CSRC = os.path.join(os.path.dirname(HERE), "gputimeseriescompressionoptimizer_amd", "csrc")


def test_contexts_that_share_give_back_their_cached_blocks(tmp_path):
    exe = str(tmp_path / "allocator")
    subprocess.run(["g++", "-std=c++17", "-O1", "-D__HIP_PLATFORM_AMD__",
                    "-I/opt/rocm/include", os.path.join(HERE, "cpp", "allocator.cpp"),
                    os.path.join(CSRC, "allocator.cpp"), "-o", exe, "-pthread"], check=True)
    r = subprocess.run([exe], capture_output=True, text=True, timeout=60)
    assert r.returncode == 0 and r.stdout == "ok\n", r.stderr
