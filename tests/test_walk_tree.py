"""The host builder of the walk tree (tests/native/walk_tree_check.cpp, built and run here)."""
import os
import subprocess

ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))
CSRC = os.path.join(ROOT, "sort_amd", "csrc")


def test_walk_tree_invariants(tmp_path):
    exe = str(tmp_path / "walk_tree_check")
    subprocess.run(["g++", "-O2", "-std=c++17", "-ffp-contract=off", "-pthread", "-I", CSRC, "-o", exe,
                    os.path.join(ROOT, "tests", "native", "walk_tree_check.cpp"), os.path.join(CSRC, "bvh_build.cpp"),
                    os.path.join(CSRC, "walk_tree.cpp")], check=True)
    r = subprocess.run([exe], capture_output=True, text=True, timeout=120)
    assert r.returncode == 0 and r.stdout.strip() == "ok", r.stdout + r.stderr
