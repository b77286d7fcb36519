"""The 3D transform over mesh lengths of every radix, of one, two and three
stages, and with prime factors above 7: SPME forces and energies of a few
charges against the oracle, and MC reciprocal deltas from the kept
spectrum."""
import numpy as np
import pytest

import oracle as O
from molsim_amd import engine as E
from helpers import rel_rms

pytestmark = pytest.mark.gpu

EFP = E.epsi0_four_pi() / 78.4

# (s1, s2 = s3): the reference, and so the oracle, takes s3 for the y axis
MESHES = [(16, 14), (8, 12), (10, 16), (18, 20), (20, 24), (28, 36), (24, 30), (32, 40), (40, 64),
          (42, 48), (50, 54), (60, 70), (72, 80), (84, 90), (108, 18), (16, 108), (112, 28),
          (16, 112), (20, 128), (96, 100), (128, 10), (12, 150), (140, 16), (126, 42), (18, 126),
          (16, 180), (180, 20), (200, 14), (8, 200), (252, 16), (12, 240), (256, 16), (8, 256),
          (512, 16), (8, 512), (1024, 16), (8, 1024), (22, 32), (32, 22), (36, 26), (44, 34)]


def setup(mesh, n, prec):
    mesh = np.array([mesh[0], mesh[1], mesh[1]])
    box = 1.2 * mesh
    rng = np.random.default_rng(int(mesh.sum()))
    m = np.maximum((box / 2.0).astype(int), 1)
    site = rng.choice(m.prod(), n, replace=False)
    ro = np.stack([site // (m[1] * m[2]), site // m[2] % m[1], site % m[2]], 1) + 0.5
    ro = ro * (box / m) - box / 2 + rng.uniform(-0.6, 0.6, (n, 3))
    types = (1 + np.arange(n) % 2).astype(np.int32)
    zat = np.array([1.0, -1.0])
    # no pair within the tables' 0.5 A: the reciprocal part alone
    tab = E.build_tables(zat, np.array([0.3, 0.3]), np.array([1.0, 1.0]), rcut=0.5,
                         epsi_four_pi=EFP, alpha=0.45)
    eng = E.ForceEngine(n, prec)
    eng.set_box(box)
    eng.set_particles(types, zat[types - 1], np.ones(2))
    eng.set_tables(tab, 0.5)
    eng.set_ewald("spm", 0.45, 4, mesh, 0, False, False, EFP)
    eng.set_neighbor("vlist", 1.0, 0)
    eng.upload_positions(ro)
    orc = O.Oracle(box, types, zat[types - 1], O.Tables(tab.ubuf, tab.iubuflow, tab.nugrid,
                   tab.r2umin, None), 0.5, ewald="spm", alpha=0.45, epsi_four_pi=EFP, order=4,
                   mesh=tuple(int(v) for v in mesh), drnlist=1.0, maxnneigh=n)
    return eng, orc, ro, box


# FP64: summation order; mixed: FP32 spreading, transforms and gather, some
# ten roundings of 2^-24 per value.  Energies relative to the mesh sum: u%rec
# is that sum minus the self term, nearly as large for these charges.
@pytest.mark.parametrize("prec,ftol,etol", [("fp64", 1e-10, 1e-11), ("mixed", 1e-5, 1e-6)])
@pytest.mark.parametrize("mesh", MESHES, ids=lambda m: "x".join(map(str, m)))
def test_spme_over_mesh_lengths(mesh, prec, ftol, etol):
    if prec == "mixed" and max(mesh) > 512:
        pytest.skip("FP32's force error grows with the length: 1-2e-5 here, on any FFT")
    eng, orc, ro, box = setup(mesh, 60, prec)
    f, en = eng.utotal()
    orc.set_list(ro)
    fo, eo = orc.utotal(ro)
    assert rel_rms(f, fo) <= ftol
    mesh_sum = eo["rec"] + EFP * 0.45 / np.sqrt(np.pi) * ro.shape[0]
    assert abs(en.rec - eo["rec"]) <= etol * mesh_sum
    assert abs(en.virial - eo["virial"]) <= 10 * etol * mesh_sum
    # a trial move from the kept spectrum (transformed along z alone)
    new = ro.copy()
    new[7] = np.clip(ro[7] + np.array([0.4, -0.3, 0.2]), -box / 2, box / 2)
    du = eng.mc_delta_rec([8], new[7:8])
    _, en_new = orc.utotal(new)
    assert abs(du - (en_new["rec"] - eo["rec"])) <= etol * mesh_sum
    eng.close()
