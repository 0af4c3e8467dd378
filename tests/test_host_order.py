"""The host side of the library without a GPU (tests/cpp/host_order.cpp): what it enqueues, on which stream,
and which launches wait for which others.  The program is compiled from pl_api.cpp and a record of the HIP
calls and launches in the place of the runtime and the kernels."""
import os
import subprocess

import pytest

from conftest import ROOT

from permutohedral_lattice_amd import build as hip_build

SCENARIOS = ["read_on_the_own_stream", "replay_on_the_own_stream", "one_stream_for_all", "handle_given_out_again",
             "two_callers_and_builds", "changing_company", "own_stream_captured", "failed_blur", "no_pointer_kept",
             "failed_batch", "batches_either_way", "more_rows_of_sums"]


@pytest.fixture(scope="module")
def host_order(tmp_path_factory):
    out = tmp_path_factory.mktemp("host_order")
    csrc = os.path.join(ROOT, "permutohedral_lattice_amd", "csrc")
    objects = []
    for source in (os.path.join(csrc, "pl_api.cpp"), os.path.join(ROOT, "tests", "cpp", "host_order.cpp")):
        objects.append(str(out / (os.path.basename(source) + ".o")))
        subprocess.run([hip_build.hipcc(), "-O1", "-std=c++17", "--offload-arch=gfx950", "--offload-host-only",
                        "-x", "hip", "-I" + os.path.join(ROOT, "include"), "-I" + csrc, "-c", source,
                        "-o", objects[-1]], check=True)
    binary = str(out / "host_order.bin")
    # (launches that no scenario reaches are left out of the program)
    subprocess.run(["g++", "-no-pie"] + objects + ["-Wl,--unresolved-symbols=ignore-all", "-o", binary], check=True)
    return binary


@pytest.mark.parametrize("scenario", SCENARIOS)
def test_what_the_host_enqueues(host_order, scenario):
    res = subprocess.run([host_order, scenario], stdout=subprocess.PIPE, stderr=subprocess.STDOUT, text=True, timeout=60)
    assert res.returncode == 0, res.stdout
