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
seen, grids = [], 0
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
        assert all(need <= room for need, room in seen), (kmax, prec, seen)
        L.mdffgpu_destroy(h)
        grids += bool(seen)
        print(kmax, prec, seen, flush=True)
assert grids >= 15, grids  # the others take the direct sums
""")


# A call that has to grow the grid's tile lists: the displacement test asks for
# a rebuild and the entries of the lists come out as GROWN; with `fail` the allocation
# after it is refused.
GROW = """
import ctypes, host_hip as H
import numpy as np
from mdff_amd import configs as C, params as P
names, arm, fail = [], set(), lambda n: False
mesh = []
def launch(name, gx, gy, gz, args):
    names.append(name)
    if b"k_rho_reduce64" in name:
        mesh.append(H.pointer(args, 0, 24))
    if b"k_disp" in name and "disp" in want:
        arm.add("disp")
    if b"k_grid_cap" in name and "cap" in want:
        arm.add("cap")
def d2h(dst, n):
    if n == 8 and "cap" in arm:
        arm.discard("cap")
        ctypes.c_longlong.from_address(dst).value = GROWN
    elif n == 8 and "disp" in arm:
        arm.discard("disp")
        ctypes.memset(dst, 0x41, n)
def refuse(n, kind):
    return 1 if fail(n) and kind == 0 and any(b"k_grid_cap" in x for x in names) else 0
want, GROWN = set(), 100000
H.hooks(launch=launch, refuse=refuse, d2h=d2h)
L = H.lib()
"""


def test_context_after_a_refused_bin_allocation(host_hip):
    """The evaluation goes on with the direct sums, the phases of which it
    makes, and so do the next ones; nothing reads the lists."""
    host_hip(GROW + """
# the lists alone are refused, or every allocation after the bins: then the
# first call reports it and the next one makes what the direct sums need
for all_of_them, prec, direct in ((f, *w) for f in (False, True) for w in (
        (P.PREC_FP64, b"k_rho64"), (P.PREC_MIXED, b"mx_rho"))):
    s = C.silica(20, 40, seed=8, rc=4.0, kmax=10, pim=False)
    s.params.precision = prec
    st, h = H.create(L, s)
    assert st == 0
    assert H.engforce_device(L, h, s.r) == 0
    assert any(b"k_grid_lists" in x for x in names)
    del names[:]
    want.update(("disp", "cap"))
    del mesh[:]
    fail = lambda n: all_of_them or n == 8 * (GROWN + GROWN // 8 + 8)
    st = H.engforce_device(L, h, s.r)
    assert (st != 0) == all_of_them, (prec, st)
    assert any(b"k_grid_cap" in x for x in names)
    assert not any(b"k_grid_lists" in x for x in names)
    fail = lambda n: False
    want.clear()
    for again in range(2):
        if all_of_them or again:
            del names[:]
            assert H.engforce_device(L, h, s.r) == 0
        assert any(direct in x for x in names), names
        if prec == P.PREC_FP64:
            assert mesh and all(mesh), mesh  # A_k of k_rho_reduce64
        if not all_of_them and not again:
            bins = max(k for k, x in enumerate(names) if b"k_grid_cap" in x)
            assert any(b"k_prepare" in x for x in names[bins:])
        else:
            assert not any(b"k_grid" in x for x in names), names
    L.mdffgpu_destroy(h)
""")


def test_context_without_memory_for_the_grid(host_hip):
    """Every allocation of a creation refused in turn: those of the grid leave
    a context that takes the direct sums, the others an error."""
    host_hip(GROW + """
left = [0]
def refuse_nth(n, kind):
    left[0] -= 1
    return 1 if left[0] == 0 else 0
H.hooks(launch=launch, refuse=refuse_nth)
for prec, direct in ((P.PREC_FP64, b"k_rho64"), (P.PREC_MIXED, b"mx_rho")):
    s = C.silica(20, 40, seed=8, rc=4.0, kmax=10, pim=True)
    s.params.precision = prec
    kept = 0
    for nth in range(1, 200):
        left[0] = nth
        st, h = H.create(L, s)
        if left[0] > 0:
            break
        if st:
            continue
        kept += 1
        del names[:]
        assert H.engforce_device(L, h, s.r) == 0
        assert any(direct in x for x in names) and not any(b"k_grid" in x for x in names)
        L.mdffgpu_destroy(h)
    assert st == 0 and kept >= 10, kept
    L.mdffgpu_destroy(h)
""")


def test_set_cell_without_memory_for_the_k_mesh(host_hip):
    """set_cell of a mixed grid context whose k mesh is refused reports it; the
    plan has the new cell, and the next EFG call makes the tables it reads."""
    host_hip(GROW + """
s = H.melt(60, False)
s.params.kES[:] = [6, 6, 6]
s.params.precision = P.PREC_MIXED
st, h = H.create(L, s)
assert st == 0
A = np.ascontiguousarray(1.01 * np.asarray(s.A).reshape(-1, order="F"))
for which in (1, 2, 3, 4):  # chunks, A_k and the rest in turn
    left = [which]
    def refuse_nth(n, kind):
        if kind == 0 and names and b"k_grid_factors" in names[-1]:
            left[0] -= 1
            return 1 if left[0] == 0 else 0
        return 0
    H.hooks(launch=launch, refuse=refuse_nth)
    del names[:], mesh[:]
    assert L.mdffgpu_set_cell(h, A.ctypes.data_as(H.dp)) == 3
    assert any(b"k_grid_factors" in x for x in names)
    H.hooks(launch=launch)
    assert H.engforce_device(L, h, s.r) == 0
    assert any(b"k_grid_spread" in x for x in names) and not mesh
    assert H.efg(L, h, s.r) == 0, L.mdffgpu_last_error(h)
    assert mesh and all(mesh), mesh
L.mdffgpu_destroy(h)
""")


def test_host_memory_failure_is_a_status(host_hip):
    """Without pinned memory the staging of a host call falls back to ordinary
    memory; without that too the call returns MDFFGPU_ERR_ALLOC, as do a
    context and a batch whose tables find none, and the next call works."""
    host_hip(GROW + """
from mdff_amd import _lib
_lib._lib = L
from mdff_amd.batch import Batch
s = H.melt(600, True)
s.params.kES[:] = [6, 6, 6]
st, h = H.create(L, s)
assert st == 0
assert H.engforce_device(L, h, s.r) == 0  # the numbering is decided
H.hooks(launch=launch, refuse=lambda n, kind: 1 if kind == 1 else 0)
H.hip.host_hip_new_limit(6 * 600 * 8)
assert H.engforce(L, h, s.r) == 3
assert b"host memory" in L.mdffgpu_last_error(h)
H.hip.host_hip_new_limit(2 ** 62)
assert H.engforce(L, h, s.r) == 0
H.hooks(launch=launch)
assert H.engforce(L, h, s.r) == 0
L.mdffgpu_destroy(h)
s.params.task_coul_quad[0] = 1  # direct sums
st, h = H.create(L, s)
A = np.ascontiguousarray(np.asarray(s.A).reshape(-1, order="F"))
H.hip.host_hip_new_limit(1024)
assert L.mdffgpu_set_cell(h, A.ctypes.data_as(H.dp)) == 3
H.hip.host_hip_new_limit(2 ** 62)
assert H.engforce_device(L, h, s.r) == 0
L.mdffgpu_destroy(h)
s.params.task_coul_quad[0] = 0
b = Batch.from_systems([s, s], precision=P.PREC_FP64)
r = np.ascontiguousarray(np.concatenate([s.r, s.r]).T)
H.hip.host_hip_new_limit(64)
assert L.mdffgpu_batch_set_positions(b._h, r.ctypes.data, None) == 3
H.hip.host_hip_new_limit(2 ** 62)
assert L.mdffgpu_batch_set_positions(b._h, r.ctypes.data, None) == 0
b.close()
""")


def test_fp64_grid_context_makes_no_k_mesh(host_hip):
    """Creation and set_cell neither fill nor hold the tables of the direct
    sums (3 kpad doubles of k vectors among them); a context that takes the
    direct sums, or a mixed one (whose EFG is summed in FP64), does."""
    host_hip("""
import ctypes, host_hip as H
import numpy as np
from mdff_amd import configs as C, params as P
sizes = []
def record(n, kind):
    sizes.append(n)
    return 0
H.hooks(refuse=record)
L = H.lib()
k = 20
chunks = -(-(2 * k + 1) // 16)
KC = -(-(2 * k + 1) // chunks)
kpad = (-(-k // KC) + (k + k * (2 * k + 1)) * chunks) * KC
for prec, quad, want in ((P.PREC_FP64, 0, False), (P.PREC_FP64, 1, True), (P.PREC_MIXED, 0, True)):
    s = C.silica(20, 40, seed=8, rc=4.0, kmax=k, pim=True)
    s.params.precision = prec
    s.params.task_coul_quad[0] = quad
    del sizes[:]
    st, h = H.create(L, s)
    assert st == 0
    assert L.mdffgpu_num_kvectors(h) == ((2 * k + 1) ** 3 - 1) // 2
    assert (24 * kpad in sizes) == want, (prec, quad)
    del sizes[:]
    A = np.ascontiguousarray(1.01 * np.asarray(s.A).reshape(-1, order="F"))
    assert L.mdffgpu_set_cell(h, A.ctypes.data_as(H.dp)) == 0
    assert (24 * kpad in sizes) == want, (prec, quad)
    assert H.engforce_device(L, h, s.r) == 0
    L.mdffgpu_destroy(h)
""")


def test_batch_after_a_refused_allocation(host_hip):
    """A batch whose set_positions failed refuses evaluations (its lists are
    gone) until one succeeds; without the memory for the grid it takes the
    direct sums."""
    host_hip(GROW + """
from mdff_amd import _lib
_lib._lib = L
from mdff_amd.batch import Batch
systems = [C.silica(n, 2 * n, seed=30 + n, rc=4.5, kmax=4, pim=True, pot_seed=3) for n in (16, 21)]
r = np.ascontiguousarray(np.concatenate([s.r for s in systems]).T)
tgt, loss = np.zeros_like(r), ctypes.c_double()
for prec in (P.PREC_FP64, P.PREC_MIXED):
    b = Batch.from_systems(systems, precision=prec)
    grad = np.zeros(b.nparam)
    def evaluate():
        return L.mdffgpu_batch_loss_grad(b._h, tgt.ctypes.data, None, ctypes.byref(loss),
                                         grad.ctypes.data_as(H.dp), 3, None, None, None)
    def positions():
        del names[:]
        return L.mdffgpu_batch_set_positions(b._h, r.ctypes.data, None)
    # every allocation of the first calls in turn, a batch each
    left = [0]
    def refuse_nth(n, kind):
        left[0] -= 1
        return 1 if left[0] == 0 else 0
    failed = direct = 0
    for nth in range(1, 64):
        b = Batch.from_systems(systems, precision=prec)
        H.hooks(launch=launch, refuse=refuse_nth)
        left[0] = nth
        st = positions()
        if left[0] > 0:
            break
        if st:
            failed += 1
            assert evaluate() == 1, (prec, nth)
            assert positions() == 0
            assert evaluate() == 0
        else:
            del names[:]
            assert evaluate() == 0
            if not any(b"k_grid" in x for x in names):
                direct += 1
        b.close()
    assert st == 0 and failed > 0 and direct >= 10, (failed, direct)
    assert evaluate() == 0 and any(b"k_grid_spread" in x for x in names)
    # and the growth of the lists
    H.hooks(launch=launch, refuse=refuse, d2h=d2h)
    want.add("cap")
    fail = lambda n: True
    assert positions() == 0
    fail = lambda n: False
    want.clear()
    del names[:]
    assert evaluate() == 0
    assert not any(b"k_grid" in x for x in names)
    assert positions() == 0
    assert evaluate() == 0
    b.close()
""")


# (kmax, atoms, polarizable): the path of the reciprocal sums on either side of
# the lines of the rule in FP64 and in mixed precision
ROUTES = [
    # small meshes
    ((2, 2, 2), 60, True, "direct", "grid"),
    ((3, 3, 3), 60, True, "grid", "grid"),
    # many atoms per tile
    ((5, 5, 5), 90, True, "grid", "grid"),
    ((5, 5, 5), 90, False, "direct", "grid"),
    ((5, 5, 5), 3000, True, "direct", "grid"),
    ((5, 5, 5), 3000, False, "direct", "direct"),
    ((3, 3, 3), 1500, True, "direct", "direct"),
    ((10, 10, 10), 648, False, "grid", "grid"),
    ((10, 10, 10), 3000, True, "grid", "grid"),
    ((8, 8, 8), 12288, True, "direct", "grid"),
    ((24, 24, 24), 3000, False, "grid", "grid"),
    # few atoms with a large mesh; mixed has no direct sums past 24
    ((60, 60, 60), 3, False, "direct", "grid"),
    ((60, 60, 60), 192, True, "grid", "grid"),
    ((80, 80, 80), 192, True, "direct", "grid"),
    ((10, 100, 100), 48, True, "direct", "grid"),
    ((5, 80, 80), 48, True, "grid", "grid"),
    # past the grid's extents
    ((3, 3, 115), 90, True, "direct", "direct"),
]


def test_route_of_the_reciprocal_sums(host_hip):
    host_hip(f"""
import host_hip as H
from mdff_amd import params as P
names = []
H.hooks(launch=lambda name, gx, gy, gz, args: names.append(name))
L = H.lib()
for kmax, n, pim, *want in {ROUTES!r}:
    s = H.melt(n, pim)
    s.params.kES[:] = list(kmax)
    for prec, path in zip((P.PREC_FP64, P.PREC_MIXED), want):
        s.params.precision = prec
        st, h = H.create(L, s)
        assert st == 0
        del names[:]
        assert H.engforce_device(L, h, s.r) == 0
        L.mdffgpu_destroy(h)
        grid = any(b"k_grid_spread" in x for x in names)
        direct = any(b"k_rho64" in x or b"mx_rho" in x for x in names)
        assert (grid, direct) == (path == "grid", path == "direct"), (kmax, n, pim, prec, path)
# mixed with an FP64 reciprocal space: by the FP64 lines where it has both
for k, path in ((5, b"k_rho64"), (60, b"k_grid_spread")):
    s = H.melt(3, False)
    s.params.kES[:] = [k] * 3
    s.params.precision, s.params.mixed_fp64_parts = P.PREC_MIXED, P.MIXED_FP64_KSPACE
    st, h = H.create(L, s)
    assert st == 0, k
    del names[:]
    assert H.engforce_device(L, h, s.r) == 0
    L.mdffgpu_destroy(h)
    assert any(path in x for x in names), k
""")


def test_route_of_a_mixed_batch(host_hip):
    """Either side of the lines of the rule of a mixed batch (atoms and number
    of the configurations, kmax); differing kmax take the per-k kernels."""
    host_hip("""
import copy, ctypes, host_hip as H
import numpy as np
from mdff_amd import params as P, _lib
names = []
H.hooks(launch=lambda name, gx, gy, gz, args: names.append(name))
_lib._lib = L = H.lib()
from mdff_amd.batch import Batch
for natm, nconf, kmax, prec, want in (
        (96, 4, 8, P.PREC_MIXED, "grid"), (96, 64, 8, P.PREC_MIXED, "direct"),
        (399, 16, 8, P.PREC_MIXED, "grid"), (399, 64, 8, P.PREC_MIXED, "direct"),
        (96, 10, 12, P.PREC_MIXED, "direct"), (399, 1, 3, P.PREC_MIXED, "grid"),
        (1800, 2, 3, P.PREC_MIXED, "direct"), (96, 64, 8, P.PREC_FP64, "grid"),
        (1800, 2, 3, P.PREC_FP64, "grid"), (96, 2, (5, 6), P.PREC_MIXED, "per k"),
        (96, 2, (5, 6), P.PREC_FP64, "per k")):
    ks = kmax if isinstance(kmax, tuple) else (kmax,) * nconf
    s0 = H.melt(natm, True)
    systems = [copy.deepcopy(s0) for k in ks]
    for s, k in zip(systems, ks):
        s.params.kES[:] = [k] * 3
    b = Batch.from_systems(systems, precision=prec)
    r = np.ascontiguousarray(np.concatenate([s.r for s in systems]).T)
    tgt, loss, grad = np.zeros_like(r), ctypes.c_double(), np.zeros(b.nparam)
    assert L.mdffgpu_batch_set_positions(b._h, r.ctypes.data, None) == 0
    del names[:]
    assert L.mdffgpu_batch_loss_grad(b._h, tgt.ctypes.data, None, ctypes.byref(loss),
                                     grad.ctypes.data_as(H.dp), 3, None, None, None) == 0
    # the reverse pass spreads with k_grid_spread_adj
    got = [w for w, key in (("grid", b"13k_grid_spreadI"), ("direct", b"mx_rho"),
                            ("per k", b"k_b_rho")) if any(key in x for x in names)]
    assert got == [want], (natm, nconf, kmax, prec, got)
    assert any(b"k_b_rev_dir" in x for x in names) == (want != "per k")
    b.close()
""")
