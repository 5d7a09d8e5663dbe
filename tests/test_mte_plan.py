"""The FP32 MTE launch plan on the host (CPU): the header that the launches use
(mte_plan.h) built into a host program."""
import pathlib
import subprocess

REPO = pathlib.Path(__file__).resolve().parent.parent


def test_plan_of_rows_and_waves(tmp_path):
    exe = tmp_path / "mte_plan_check"
    subprocess.run(["g++", "-O1", "-std=c++17", "-I", str(REPO / "transportoptimiser_amd/csrc"),
                    "-I", str(REPO / "include"),
                    str(REPO / "tests/native/mte_plan_check.cpp"), "-o", str(exe)],
                   check=True, capture_output=True, text=True)
    r = subprocess.run([str(exe)], capture_output=True, text=True, timeout=60)
    assert r.returncode == 0, r.stdout
