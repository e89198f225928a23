"""The batch's choice between narrow and wide workgroups (cuopt_amd/csrc/batch_width.hpp), compiled
with g++ beside a check program (tests/width_check/width_check.cpp): batches that were
measured in both widths get the faster one."""

import os
import subprocess

ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))


def test_measured_batches_get_the_faster_width(tmp_path):
    exe = str(tmp_path / "width_check")
    r = subprocess.run(["g++", "-std=c++17", "-O1", "-Wall", "-Werror", "-I" + os.path.join(ROOT, "cuopt_amd", "csrc"),
                        os.path.join(ROOT, "tests", "width_check", "width_check.cpp"), "-o", exe],
                       capture_output=True, text=True)
    assert r.returncode == 0, r.stderr
    r = subprocess.run([exe], capture_output=True, text=True, timeout=60)
    assert r.returncode == 0 and "OK" in r.stdout, r.stdout + r.stderr
