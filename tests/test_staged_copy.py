"""The host side of the staged copies under ThreadSanitizer (CPU): bytes arrive,
errors end the copy, and no access of its threads races with another."""
import os
import shutil
import subprocess

import pytest

ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))

pytestmark = pytest.mark.skipif(shutil.which("g++") is None, reason="no host compiler")


def test_ring_of_host_copies(tmp_path):
    exe = str(tmp_path / "staged")
    r = subprocess.run(["g++", "-std=c++17", "-O1", "-g", "-fsanitize=thread", "-pthread",
                        os.path.join(ROOT, "tests/sanitize/staged_main.cpp"), "-o", exe],
                       capture_output=True, text=True)
    assert r.returncode == 0, r.stderr[-3000:]
    r = subprocess.run([exe], capture_output=True, text=True, timeout=110,
                       env=dict(os.environ, TSAN_OPTIONS="halt_on_error=1"))
    if "unexpected memory mapping" in r.stderr:
        pytest.skip("ThreadSanitizer cannot map its memory here")
    assert "data race" not in r.stderr, r.stderr[-4000:]
    assert r.returncode == 0 and "staged copies passed" in r.stdout, r.stdout + r.stderr[-2000:]
