"""CPU: the order between trees and multi-tree launches, followed through the
events the library records and waits for (tests/cpp/batch_events.cpp, linked
against the emulation build)."""
import os
import shutil
import subprocess

import pytest

HERE = os.path.dirname(os.path.abspath(__file__))
EMU = os.path.join(HERE, "cpu_emu")


@pytest.fixture(scope="module")
def exe(tmp_path_factory):
    if shutil.which("g++") is None:
        pytest.skip("g++ is not available")
    if os.environ.get("LD_PRELOAD"):
        pytest.skip("AddressSanitizer executables need their runtime first; a preloaded library is present")
    subprocess.run(["make", "-s", "-C", EMU], check=True)
    out = tmp_path_factory.mktemp("batch_events") / "batch_events"
    subprocess.run(["g++", "-std=c++20", "-O1", "-g", "-fsanitize=address", "-include", os.path.join(EMU, "hip_emu.h"),
                    "-I", EMU, "-I", os.path.join(HERE, "..", "include"), os.path.join(HERE, "cpp", "batch_events.cpp"),
                    "-o", str(out), "-L", EMU, "-likd_emu", f"-Wl,-rpath,{EMU}", "-lpthread"], check=True)
    return out


@pytest.mark.parametrize("scenario", ["two_batches", "captured_launch", "closed_batches"])
def test_order_between_launches_and_trees(exe, scenario):
    r = subprocess.run([str(exe), scenario], capture_output=True, text=True, timeout=300,
                       env=dict(os.environ, ASAN_OPTIONS="detect_leaks=0"))
    assert r.returncode == 0, r.stdout[-2000:] + r.stderr[-3000:]
    assert r.stdout.startswith("ok")
