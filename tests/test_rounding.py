"""The embedding's substitutes for divisions, compiled for the host (tests/cpp/rounding.cpp), against the divisions."""
import os
import subprocess

from conftest import ROOT

from permutohedral_lattice_amd import build as hip_build


def test_they_round_as_the_divisions_do(tmp_path):
    binary = str(tmp_path / "rounding.bin")
    subprocess.run([hip_build.hipcc(), "-O2", "-std=c++17", "--offload-arch=gfx950", "--offload-host-only",
                    "-ffp-contract=off", "-x", "hip", "-I" + os.path.join(ROOT, "include"),
                    "-I" + os.path.join(ROOT, "permutohedral_lattice_amd", "csrc"),
                    os.path.join(ROOT, "tests", "cpp", "rounding.cpp"), "-o", binary], check=True)
    res = subprocess.run([binary], stdout=subprocess.PIPE, stderr=subprocess.STDOUT, text=True, timeout=120)
    assert res.returncode == 0, res.stdout
