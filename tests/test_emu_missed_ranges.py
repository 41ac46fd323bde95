"""CPU: the kNN walk a tree takes while its stored ranges may miss points, and the
one it takes again when the whole tree has been rebuilt (emulation build)."""
import os
import shutil
import subprocess

import pytest

HERE = os.path.dirname(os.path.abspath(__file__))
EMU = os.path.join(HERE, "cpu_emu")


def test_walk_after_restores_and_rebuilds(tmp_path):
    if shutil.which("g++") is None:
        pytest.skip("g++ is not available")
    if os.environ.get("LD_PRELOAD"):
        pytest.skip("AddressSanitizer executables need their runtime first; a preloaded library is present")
    subprocess.run(["make", "-s", "-C", EMU], check=True)
    exe = tmp_path / "missed_ranges"
    subprocess.run(["g++", "-std=c++20", "-O1", "-g", "-fsanitize=address", "-I", os.path.join(HERE, "..", "include"),
                    os.path.join(HERE, "cpp", "missed_ranges.cpp"), "-o", str(exe), "-L", EMU, "-likd_emu",
                    f"-Wl,-rpath,{EMU}", "-lpthread"], check=True)
    r = subprocess.run([str(exe)], capture_output=True, text=True, timeout=300,
                       env=dict(os.environ, ASAN_OPTIONS="detect_leaks=0"))
    assert r.returncode == 0, r.stdout[-2000:] + r.stderr[-3000:]
    assert r.stdout.startswith("ok")
