"""The batch's conjugate gradient kernels on a CPU model of workgroups (tests/host/model): a
set that breaks down keeps its iterate whatever the order in which wavefronts see its flag,
and only a solved set is left with the flag of one."""
import os
import subprocess

ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))
CSRC = os.path.join(ROOT, "cardiomechanics_amd", "csrc")


def test_breakdown_and_flags(tmp_path):
    exe = tmp_path / "cg_breakdown"
    subprocess.check_call(["g++", "-O1", "-std=c++17", "-pthread", "-Wno-unknown-pragmas", "-x", "c++",
                           os.path.join(ROOT, "tests", "host", "cg_breakdown.cpp"),
                           "-I", os.path.join(ROOT, "tests", "host", "model"), "-I", CSRC,
                           "-I", os.path.join(ROOT, "include"), "-o", str(exe)])
    out = subprocess.run([str(exe)], capture_output=True, text=True, timeout=120)
    print(out.stdout)
    assert out.returncode == 0, out.stdout + out.stderr
