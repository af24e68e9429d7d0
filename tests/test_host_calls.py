"""Host code of the library without a GPU: the HIP runtime is a stand-in
whose kernels do not run (host_hip.cpp), so that allocations, their failures
and the launches with their arguments can be looked at.  Each test runs in a
process of its own."""
import os
import subprocess
import sys

import pytest

from mdff_amd import _lib

HERE = os.path.dirname(os.path.abspath(__file__))
pytestmark = pytest.mark.skipif(not os.path.exists(_lib.LIB_PATH),
                                reason="libmdffgpu.so not built")


@pytest.fixture(scope="module")
def host_hip(tmp_path_factory):
    so = str(tmp_path_factory.mktemp("host_hip") / "libhost_hip.so")
    subprocess.run(["g++", "-O1", "-std=c++17", "-shared", "-fPIC", "-o", so,
                    os.path.join(HERE, "host_hip.cpp")], check=True)

    def run(code):
        env = dict(os.environ, HOST_HIP=so)
        env["PYTHONPATH"] = os.pathsep.join([HERE, os.path.dirname(HERE)])
        r = subprocess.run([sys.executable, "-c", code], env=env, stdout=subprocess.PIPE,
                           stderr=subprocess.STDOUT, text=True, timeout=300)
        assert r.returncode == 0, r.stdout
        return r.stdout

    return run


def test_energy_partials_of_the_grid_fit_their_buffer(host_hip):
    """The final Ewald call writes seven partials per eight (n2, n3) columns,
    whatever the first axis: thin cells with few atoms need the most room
    next to the sums that the buffer is otherwise sized for."""
    host_hip("""
import ctypes, host_hip as H
from mdff_amd import configs as C, params as P
seen = []
def launch(name, gx, gy, gz, args):
    if b"k_grid_midILb1E" in name:
        # EnArgs: cell (19 doubles), alpha, pout
        room = H.hip.host_hip_room(H.pointer(args, 4, 160))
        seen.append((7 * 8 * gx, room))
H.hooks(launch=launch)
L = H.lib()
for kmax in ((1, 1, 1), (1, 58, 58), (2, 58, 58), (1, 64, 64), (2, 80, 80), (5, 80, 80),
             (7, 114, 114), (1, 114, 114), (114, 1, 1), (12, 12, 12)):
    for prec in (P.PREC_FP64, P.PREC_MIXED):
        s = C.silica(20, 40, seed=8, rc=4.0, kmax=3, pim=True)
        s.params.kES[:] = list(kmax)
        s.params.precision = prec
        st, h = H.create(L, s)
        assert st == 0, kmax
        del seen[:]
        assert H.engforce_device(L, h, s.r) == 0
        assert seen and all(need <= room for need, room in seen), (kmax, prec, seen)
        L.mdffgpu_destroy(h)
        print(kmax, prec, seen, flush=True)
""")
