"""Device blocks of the contexts (csrc/blocks.h) on the CPU, over a device of limited capacity: the
model is tests/blocks_model.cpp, run plain and under ThreadSanitizer; it stops at its first
failure."""
import os
import shutil
import subprocess

import pytest

ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))
SRC = os.path.join(ROOT, "tests", "blocks_model.cpp")
INC = os.path.join(ROOT, "accmultiwayjoins_amd", "csrc")


@pytest.mark.skipif(shutil.which("g++") is None, reason="needs g++")
@pytest.mark.parametrize("flags", [["-O2", "-Wall"], ["-O1", "-g", "-fsanitize=thread"]],
                         ids=["plain", "tsan"])
def test_blocks(tmp_path, flags):
    exe = str(tmp_path / "blocks_model")
    try:
        subprocess.check_call(["g++", "-std=c++17", "-pthread", "-I", INC, *flags, SRC, "-o", exe])
    except subprocess.CalledProcessError:
        if "-fsanitize=thread" not in flags:
            raise
        pytest.skip("ThreadSanitizer is not available to g++ here")
    out = subprocess.run([exe], capture_output=True, text=True, timeout=300)
    assert out.returncode == 0, out.stderr[-4000:] + out.stdout
    assert "ThreadSanitizer" not in out.stderr, out.stderr[-4000:]
    assert out.stdout.strip().endswith("OK")
