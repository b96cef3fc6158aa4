"""Kernels on a CPU model of workgroups (tests/host/model), where a test chooses the order in which
wavefronts run.  cg_breakdown: the batch's conjugate gradient; a set that breaks down keeps
its iterate whatever the order in which wavefronts see its flag, and only a solved set is left
with the flag of one.  bicgstab: the whole solver with block Jacobi."""
import os
import subprocess

import pytest

ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))
CSRC = os.path.join(ROOT, "cardiomechanics_amd", "csrc")


@pytest.mark.parametrize("program", ["cg_breakdown", "bicgstab"])
def test_kernels_on_the_workgroup_model(program, tmp_path):
    exe = tmp_path / program
    subprocess.check_call(["g++", "-O1", "-std=c++17", "-pthread", "-D__HIPCC__", "-Wno-unknown-pragmas", "-x", "c++",
                           os.path.join(ROOT, "tests", "host", program + ".cpp"),
                           "-I", os.path.join(ROOT, "tests", "host", "model"), "-I", CSRC,
                           "-I", os.path.join(ROOT, "include"), "-o", str(exe)])
    out = subprocess.run([str(exe)], capture_output=True, text=True, timeout=120)
    print(out.stdout)
    assert out.returncode == 0, out.stdout + out.stderr
