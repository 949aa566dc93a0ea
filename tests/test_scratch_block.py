"""The growth of a thread's scratch (jitnn_amd/csrc/scratch.h), driven on the CPU with an allocator that keeps books."""
import subprocess
from pathlib import Path

ROOT = Path(__file__).resolve().parent.parent


def test_scratch_block(tmp_path):
    exe = tmp_path / "scratch_block_test"
    subprocess.run(["g++", "-std=c++17", "-Wall", "-Werror", "-I", str(ROOT / "jitnn_amd" / "csrc"),
                    str(ROOT / "tests" / "scratch_block_test.cpp"), "-o", str(exe)], check=True)
    done = subprocess.run([str(exe)], capture_output=True, text=True, timeout=60)
    assert done.returncode == 0, done.stdout + done.stderr
