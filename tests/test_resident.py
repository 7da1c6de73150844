"""Host side of the resident solves (csrc/resident.h), compiled with g++ and
run here: which states count as a finished solve."""
import ctypes as C
import subprocess

import pytest

from conftest import ROOT

SRC = r"""
#include "resident.h"
extern "C" int done(int stop, int gave_up) { return xcal::resident_done(stop, gave_up); }
"""


@pytest.fixture(scope="module")
def host(tmp_path_factory):
    d = tmp_path_factory.mktemp("resident")
    (d / "host.cpp").write_text(SRC)
    so = d / "host.so"
    subprocess.run(["g++", "-std=c++17", "-shared", "-fPIC", "-Wall", "-Werror",
                    f"-I{ROOT / 'xcalibre.jl_amd' / 'csrc'}", str(d / "host.cpp"), "-o", str(so),
                    "-lpthread"], check=True)
    return C.CDLL(str(so))


@pytest.mark.parametrize("stop,gave_up,done", [
    (0, 0, 0),  # still running
    (0, 1, 0),  # given up before the end
    (1, 0, 1), (2, 0, 1), (3, 0, 1), (4, 0, 1),  # solved, itmax, breakdown, zero rhs
    # given up by one workgroup at the meeting where the others finished: its
    # rows of the solution are missing
    (1, 1, 0), (2, 1, 0), (3, 1, 0),
])
def test_a_given_up_solve_never_counts_as_finished(host, stop, gave_up, done):
    assert host.done(stop, gave_up) == done
