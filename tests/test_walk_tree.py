"""The host builder of the walk tree (programs of tests/native, built and run here)."""
import os
import subprocess

ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))
CSRC = os.path.join(ROOT, "sort_amd", "csrc")


def _run(tmp_path, name):
    exe = str(tmp_path / name)
    subprocess.run(["g++", "-O2", "-std=c++17", "-ffp-contract=off", "-pthread", "-Wno-unknown-pragmas", "-I", CSRC,
                    "-I", os.path.join(ROOT, "tests", "native", "host_hip"), "-o", exe, os.path.join(ROOT, "tests", "native", name + ".cpp"), os.path.join(CSRC, "bvh_build.cpp"),
                    os.path.join(CSRC, "walk_tree.cpp")], check=True)
    r = subprocess.run([exe], capture_output=True, text=True, timeout=120)
    assert r.returncode == 0 and r.stdout.strip() == "ok", r.stdout + r.stderr


def test_walk_tree_invariants(tmp_path):
    _run(tmp_path, "walk_tree_check")


def test_no_triangle_record_holds_a_nan(tmp_path):
    _run(tmp_path, "walk_tree_nan_check")


def test_a_walk_reaches_every_triangle_that_decides(tmp_path):
    _run(tmp_path, "walk_complete_check")


def _run_with_hip_headers(tmp_path, name, sources):
    exe = str(tmp_path / name)
    subprocess.run(["g++", "-O2", "-std=c++17", "-ffp-contract=off", "-pthread", "-D__HIP_PLATFORM_AMD__", "-I", CSRC,
                    "-I", "/opt/rocm/include", "-o", exe, os.path.join(ROOT, "tests", "native", name + ".cpp")] +
                   [os.path.join(CSRC, s) for s in sources], check=True)
    r = subprocess.run([exe], capture_output=True, text=True, timeout=120)
    assert r.returncode == 0 and r.stdout.strip() == "ok", r.stdout + r.stderr


def test_memory_short_of_a_walk_tree(tmp_path):
    _run_with_hip_headers(tmp_path, "walk_memory_check", ["bvh_build.cpp", "walk_tree.cpp", "accel_device.cpp", "pool.cpp"])


def test_rules_of_the_traversal_order(tmp_path):
    _run_with_hip_headers(tmp_path, "order_rules_check", [])
