"""Reciprocal sums through the uniform grid (grid.hip) against the oracle,
which sums every k vector: kmax from 1 (a grid of one tile, as wide as the
kernel; in FP64 by a batch, a single configuration takes the direct sums up
to about kmax 2) over odd and unequal values to a padded last tile, atoms on the cell
faces and outside the cell, a cluster (every atom in a few bins), and atoms
moved within the list's skin since their bins were made.

Tolerances: the FP64 bar of the parity tests (1e-10 of the largest value);
in mixed precision 4e-6 of the RMS, about eight times the FP32 error of the
whole evaluation.
"""
import copy

import numpy as np
import pytest

from helpers import compare_engforce
from test_gpu_geometry import skewed_silica

from mdff_amd import configs as C
from mdff_amd import params as P

pytestmark = pytest.mark.gpu

KMAX = [(1, 1, 1), (2, 5, 1), (7, 3, 12), (17, 4, 9), (4, 16, 15)]


def _edge_positions(s):
    """The melt with atoms on the faces, just inside and outside the cell."""
    r = s.r.copy()
    frac = r @ np.linalg.inv(s.A).T
    frac -= (frac[0, 0], frac[1, 1], frac[2, 2])
    frac[1, 1] = 1.0
    frac[2, 2] = -1e-17
    frac[4] += (1.0, -2.0, 3.0)
    return frac @ s.A.T


@pytest.mark.parametrize("kmax", KMAX)
@pytest.mark.parametrize("precision", [P.PREC_FP64, P.PREC_MIXED])
def test_grid_sums_match_oracle(oracle_lib, kmax, precision):
    from mdff_amd.field import ForceField
    s = skewed_silica(24, 48, seed=5, kmax=kmax, rc=4.5)
    r = _edge_positions(s)
    p = copy.deepcopy(s.params)
    p.precision = precision
    print(f"kmax {kmax} precision {precision}", flush=True)
    ff = ForceField(p, s.itype, s.A)
    orc = oracle_lib.Oracle(s.params, s.itype, s.A)
    step = 0.05 * np.random.default_rng(1).uniform(-1, 1, r.shape)
    for k in range(3):
        # the second and third frame stay within the skin of the first
        g = ff.engforce(r + k * step, itime=k + 1)
        o = orc.engforce(r + k * step, itime=k + 1)
        if precision == P.PREC_FP64:
            compare_engforce(g, o)
            continue
        for key in ("f", "mu", "ef", "efg"):
            err = np.linalg.norm(g[key] - o[key]) / np.linalg.norm(o[key])
            assert err < 4e-6, (key, err)
    assert ff.list_info()["builds"] == 1
    ff.close()


def test_grid_thin_mesh_matches_oracle(oracle_lib):
    """kmax (1, 64, 64): the final call's energy partials (one set per eight
    (n2, n3) columns) outnumber every other user of their buffer."""
    from mdff_amd.field import ForceField
    s = skewed_silica(24, 48, seed=6, kmax=(1, 64, 64), rc=4.5)
    ff = ForceField(s.params, s.itype, s.A)
    g = ff.engforce(s.r, itime=1)
    ff.close()
    compare_engforce(g, oracle_lib.Oracle(s.params, s.itype, s.A).engforce(s.r, itime=1))


def test_grid_clustered_atoms(oracle_lib):
    """All atoms in one corner of a large cell: a few bins hold everything."""
    from mdff_amd.field import ForceField
    s = C.silica(20, 40, seed=8, rc=4.0, kmax=9, pim=False, efg=True)
    A = 4.0 * s.A
    p = copy.deepcopy(s.params)
    p.cutlongrange = p.cutshortrange = 4.0
    ff = ForceField(p, s.itype, A)
    g = ff.engforce(s.r, itime=1)
    ff.close()
    compare_engforce(g, oracle_lib.Oracle(p, s.itype, A).engforce(s.r, itime=1))


def test_grid_lists_of_a_droplet_take_the_memory_of_its_atoms():
    """1,800 atoms in one corner of a cell of 13,500 tiles.  An atom is a
    candidate of at most 4 x 5 x 5 tiles (support and skin over tiles of 16 x
    8 x 8 points), 8 bytes each: 1.4 MB, and the neighbour list and pair tables
    of at most 1,800 entries per row.  Room for the longest list in every
    tile would be 190 MB."""
    import torch
    from mdff_amd.field import ForceField
    s = C.silica(600, 1200, seed=8, rc=4.0, kmax=9, pim=False)
    A = 6.0 * s.A
    s.params.kES[:] = [60, 60, 60]
    ff = ForceField(s.params, s.itype, A)
    free0 = torch.cuda.mem_get_info()[0]
    g = ff.engforce(s.r, itime=1)
    used = free0 - torch.cuda.mem_get_info()[0]
    ff.close()
    assert np.isfinite(g["f"]).all()
    assert used < 64 << 20, used


def test_grid_batch_matches_oracle(oracle_lib):
    """FP64 batch with a common, unequal-axes kmax (one plan over uneven
    configurations) against the oracle, configuration by configuration, and
    with different kmax (the per-k kernels)."""
    import torch
    from mdff_amd.batch import Batch
    systems = [C.silica(n, 2 * n, seed=30 + n, rc=4.5, kmax=4, pim=True, scf_tol=1e-12,
                        pot_seed=3) for n in (16, 21, 40)]
    for kmaxes in ([(3, 5, 4)] * 3, [(1, 1, 1)] * 3, [(2, 5, 1)] * 3,
                   [(3, 5, 4), (4, 4, 4), (3, 5, 4)]):
        for s, k in zip(systems, kmaxes):
            s.params.kES[:] = list(k)
        b = Batch.from_systems(systems, precision=P.PREC_FP64)
        b.set_positions(torch.tensor(np.concatenate([s.r for s in systems]).T.copy(),
                                     device="cuda"))
        f, _ = b.forces(0)
        f = f.cpu().numpy()
        for c, s in enumerate(systems):
            o = oracle_lib.Oracle(s.params, s.itype, s.A).engforce(s.r, itime=1)
            g = f[:, b.offsets[c]:b.offsets[c + 1]].T
            assert np.abs(g - o["f"]).max() <= 1e-10 * np.abs(o["f"]).max(), (kmaxes[c], c)
        b.close()


@pytest.mark.parametrize("precision", [P.PREC_FP64, P.PREC_MIXED])
def test_reverse_gradient_matches_tangents(precision):
    """The reverse solve (configurations with one kmax) against the tangent
    solves, which a batch takes whose kmax differ: the same configurations
    with one more whose kmax is another, subtracted out by its own batch.
    The sums differ by the rounding of the forces (FP64 1e-14, FP32 1e-6) of
    gradients whose terms cancel to a tenth."""
    import torch
    from mdff_amd.batch import Batch, get_theta
    systems = [C.silica(n, 2 * n, seed=60 + n, rc=4.5, kmax=4, pim=True, scf_tol=1e-12,
                        pot_seed=9) for n in (17, 30, 16)]
    systems[2].params.kES[:] = [5, 4, 4]
    rng = np.random.default_rng(4)

    def grads(group):
        b = Batch.from_systems(group, precision=precision)
        b.set_positions(torch.tensor(np.concatenate([s.r for s in group]).T.copy(), device="cuda"))
        n = b.natm
        target = torch.tensor(np.concatenate([tgt[id(s)] for s in group]).T.copy(), device="cuda")
        loss, grad = b.loss_grad(target, 25)
        assert len(get_theta(b.model)) == len(grad)
        b.close()
        return 3 * n * loss, 3 * n * grad

    tgt = {id(s): 10.0 * rng.standard_normal(s.r.shape) for s in systems}
    l3, g3 = grads(systems)  # tangents: the kmax differ
    l2, g2 = grads(systems[:2])  # reverse
    l1, g1 = grads(systems[2:])
    tol = 1e-10 if precision == P.PREC_FP64 else 2e-5
    assert abs(l1 + l2 - l3) <= tol * l3
    assert np.abs(g1 + g2 - g3).max() <= tol * np.abs(g3).max(), (g1 + g2, g3)
    # the electrostatic parameters, several orders smaller, on their own scale
    e = np.abs((g1 + g2 - g3)[-4:]).max()
    assert e <= 10 * tol * np.abs(g3[-4:]).max(), (g1 + g2, g3)
