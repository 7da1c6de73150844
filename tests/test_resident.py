"""Host side of the resident solves (csrc/resident.h), compiled with g++ and
run here: which states count as a finished solve, and how the solves of one
device share its compute units, in a process and between processes."""
import ctypes as C
import os
import subprocess
import sys
from concurrent.futures import ThreadPoolExecutor

import pytest

from conftest import ROOT

SRC = r"""
#include "resident.h"
static xcal::ResidentRoom room;
extern "C" {
int done(int stop, int gave_up) { return xcal::resident_done(stop, gave_up); }
void share(const char* file) { room.share(file); }
uint64_t take(int nwg, int cap) { return room.acquire(nwg, cap); }
void give(uint64_t chunks) { room.release(chunks); }
int leases(int nwg, int cap) {  // leases held at once, all given back at the end
  xcal::ResidentLease l[512];
  int n = 0;
  while (n < 512 && l[n].acquire(room, nwg, cap)) ++n;
  return n;
}
}
"""

# another process: takes room for argv[3] of 256 workgroups and says whether it
# got it, then waits for a line (argv[4] == "die": is killed holding it)
OTHER = r"""
import ctypes as C, os, signal, sys
h = C.CDLL(sys.argv[1])
h.take.restype = C.c_uint64
h.share(sys.argv[2].encode())
print(bin(h.take(int(sys.argv[3]), 256)).count("1"), flush=True)
if sys.argv[4] == "die":
    os.kill(os.getpid(), signal.SIGKILL)
sys.stdin.readline()
"""


@pytest.fixture(scope="module")
def library(tmp_path_factory):
    d = tmp_path_factory.mktemp("resident")
    (d / "host.cpp").write_text(SRC)
    so = d / "host.so"
    subprocess.run(["g++", "-std=c++17", "-shared", "-fPIC", "-Wall", "-Werror",
                    f"-I{ROOT / 'xcalibre.jl_amd' / 'csrc'}", str(d / "host.cpp"), "-o", str(so),
                    "-lpthread"], check=True)
    return so


@pytest.fixture
def host(library, tmp_path):
    """A copy of the library of its own: its room starts empty."""
    so = tmp_path / "host.so"
    so.write_bytes(library.read_bytes())
    h = C.CDLL(str(so))
    h.take.restype = C.c_uint64
    h.give.argtypes = [C.c_uint64]
    return h


def _other(library, file, nwg, how="wait"):
    p = subprocess.Popen([sys.executable, "-c", OTHER, str(library), str(file), str(nwg), how],
                         stdin=subprocess.PIPE, stdout=subprocess.PIPE, text=True)
    return p, int(p.stdout.readline())


def _end(p):
    p.communicate("\n", timeout=60)


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


@pytest.mark.parametrize("shared", [False, True])
@pytest.mark.parametrize("nwg,cap,most", [
    (256, 256, 1), (129, 256, 1), (128, 256, 2), (64, 256, 4), (4, 256, 64), (1, 256, 64),
    (257, 256, 0), (0, 256, 0), (1, 1, 1), (38, 38, 1), (13, 38, 2), (300, 304, 1),
])
def test_solves_of_one_process_fit_the_device(host, tmp_path, shared, nwg, cap, most):
    if shared:
        host.share(str(tmp_path / "room").encode())
    for _ in range(2):  # all is given back
        assert host.leases(nwg, cap) == most


def test_threads_never_hold_the_same_compute_units(host, tmp_path):
    host.share(str(tmp_path / "room").encode())

    def work(i):
        for _ in range(200):
            c = host.take(40 + 7 * i, 256)
            if c:
                with_me.append((i, c))
                held = [v for j, v in list(with_me) if j != i]
                clash = any(v & c for v in held)
                with_me.remove((i, c))
                host.give(c)
                if clash:
                    return False
        return True

    with_me = []
    with ThreadPoolExecutor(6) as ex:
        assert all(ex.map(work, range(6)))
    assert host.leases(256, 256) == 1


def test_processes_share_the_device(host, library, tmp_path):
    file = tmp_path / "room"
    host.share(str(file).encode())
    p, got = _other(library, file, 100)
    assert got == 25  # chunks of four workgroups
    q, got = _other(library, file, 200)
    assert got == 0  # refused, and nothing of it kept
    assert host.take(157, 256) == 0
    mine = host.take(156, 256)
    assert bin(mine).count("1") == 39
    _end(q)
    r, got = _other(library, file, 1)
    assert got == 0
    _end(r)
    _end(p)  # gives its part back
    assert bin(host.take(100, 256)).count("1") == 25
    host.give(mine)
    r, got = _other(library, file, 156)
    assert got == 39
    _end(r)


def test_a_killed_process_gives_its_room_back(host, library, tmp_path):
    file = tmp_path / "room"
    host.share(str(file).encode())
    p, got = _other(library, file, 256, "die")
    assert got == 64
    p.wait(timeout=60)
    assert bin(host.take(256, 256)).count("1") == 64


def test_without_the_file_a_process_counts_its_own(host, library, tmp_path):
    host.share(str(tmp_path / "no" / "such" / "folder").encode())
    p, got = _other(library, tmp_path / "no" / "such" / "folder", 256)
    assert got == 64 and host.leases(128, 256) == 2
    _end(p)


def test_a_forked_child_does_not_share_its_parents_locks(host, library, tmp_path):
    file = tmp_path / "room"
    host.share(str(file).encode())
    mine = host.take(128, 256)
    pid = os.fork()
    if pid == 0:  # what the parent holds is another process's here
        ok = host.take(256, 256) == 0 and bin(host.take(128, 256)).count("1") == 32
        os._exit(0 if ok else 1)
    assert os.waitstatus_to_exitcode(os.waitpid(pid, 0)[1]) == 0
    host.give(mine)
    assert host.leases(256, 256) == 1
