"""CPU: the branch-free box distance gives the reference's bits."""
import os
import subprocess

HERE = os.path.dirname(os.path.abspath(__file__))


def test_box_distance_equals_the_six_comparisons(tmp_path):
    exe = tmp_path / "box_distance"
    subprocess.run(["g++", "-std=c++17", "-O2", "-ffp-contract=off", "-I",
                    os.path.join(HERE, "..", "ikd-tree_amd", "csrc"), os.path.join(HERE, "cpp", "box_distance.cpp"),
                    "-o", str(exe)], check=True)
    r = subprocess.run([str(exe)], capture_output=True, text=True, timeout=120)
    assert r.returncode == 0, r.stdout
