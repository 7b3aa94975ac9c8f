"""The status with which a conjugate-gradient solve on the device ends, built
for the host under a thread sanitizer: the device's side and the host's side of
the hand-over, as two threads."""
import os
import shutil
import subprocess

import pytest

ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))


def _build(tmp_path, name, *flags):
    if shutil.which("g++") is None:
        pytest.skip("no host C++ compiler")
    exe = str(tmp_path / name)
    subprocess.run(["g++", "-O2", "-g", "-std=c++17", *flags, "-o", exe,
                    os.path.join(ROOT, "tests", "cpp", name + ".cpp"), "-pthread"],
                   check=True, timeout=120)
    return exe


def test_status_is_handed_over_in_order(tmp_path):
    exe = _build(tmp_path, "test_qs_status", "-fsanitize=thread")
    r = subprocess.run([exe], stdout=subprocess.PIPE, stderr=subprocess.STDOUT, text=True, timeout=120)
    if "FATAL: ThreadSanitizer" in r.stdout:
        pytest.skip("the sanitizer does not run on this kernel: " + r.stdout[:200])
    assert r.returncode == 0 and "0 wrong" in r.stdout and "data race" not in r.stdout, r.stdout[:3000]


def test_end_of_a_solve_is_the_host_loops(tmp_path):
    r = subprocess.run([_build(tmp_path, "test_cg_end")], stdout=subprocess.PIPE, text=True, timeout=60)
    assert r.returncode == 0 and " 0 wrong" in r.stdout, r.stdout
