"""The policy kernels' plan and row grouping on the host (CPU).

The header that the kernels compile (rovs_group.h) is built into a host program
that runs one wave's grouping over every plan of 1 to 8 controls and 64 to 512
patches, with controls drawn at random, skewed to one control and all alike:
no write outside the grouping's LDS arrays, each path once under its own
control, no more group tiles than the waves hold."""
import pathlib
import subprocess

REPO = pathlib.Path(__file__).resolve().parent.parent


def test_grouping_stays_inside_its_arrays(tmp_path):
    exe = tmp_path / "rovs_group_check"
    subprocess.run(["g++", "-O1", "-std=c++17", "-I", str(REPO / "transportoptimiser_amd/csrc"),
                    str(REPO / "tests/native/rovs_group_check.cpp"), "-o", str(exe)],
                   check=True, capture_output=True, text=True)
    r = subprocess.run([str(exe)], capture_output=True, text=True, timeout=120)
    assert r.returncode == 0, r.stdout
    # Every size of the plan was met: up to 64, 128 and 160 rows, and dense.
    assert "rows up to 64 1, 128 1, 160 1, dense 1" in r.stdout
