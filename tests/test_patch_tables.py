"""The per-cell records of the fused Vanka color step (csrc/patch_tables.cpp), on the CPU:
tests/patch_driver.cpp runs colored sweeps from the records on generated levels (cubes, open
and one-cell-wide boxes, greedy colors, Gauss-Seidel level sets, colorings that leave cells
out, rows longer than a hexahedral grid's), patches of a color in random order, and compares them with the sweep from its
definition (double sums of at most 128 terms in another order: 1e-12)."""
import shutil
import subprocess

import pytest

from conftest import ROOT


def test_sweeps_from_records(tmp_path):
    if shutil.which("g++") is None:
        pytest.skip("needs g++")
    csrc = ROOT / "to_merge_master_parmoon_amd" / "csrc"
    exe = tmp_path / "patch_driver"
    subprocess.run(["g++", "-O1", "-std=c++17", "-pthread", "-D_GLIBCXX_ASSERTIONS", f"-I{ROOT / 'include'}",
                    f"-I{csrc}", f"-I{csrc / 'problem'}", str(ROOT / "tests" / "patch_driver.cpp"),
                    str(csrc / "patch_tables.cpp"), str(csrc / "coloring.cpp"),
                    str(csrc / "problem" / "pmg_problem.cpp"), "-o", str(exe)], check=True)
    r = subprocess.run([str(exe)], capture_output=True, text=True, timeout=300)
    assert r.returncode == 0, r.stdout + r.stderr
    assert r.stdout.strip().endswith("OK"), r.stdout
    assert " 3 buffers" in r.stdout   # dofs with an odd number of updates were among them
    assert ", general," in r.stdout   # and rows longer than a hexahedral grid's
    print(r.stdout)
