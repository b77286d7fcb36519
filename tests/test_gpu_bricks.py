"""Spreading and gather over bricks of every edge (8 to 16, and larger for
meshes without such a divisor), orders 3 to 8, with empty, single and
crowded bricks, against the oracle."""
import numpy as np
import pytest

import oracle as O
from molsim_amd import engine as E
from helpers import rel_rms

pytestmark = pytest.mark.gpu

EFP = E.epsi0_four_pi() / 78.4


# mesh along x, along y and z, order, particles: brick edges 15 (order 6:
# tile planes of 20 x 20), 12, 9, 13, 11, 16, 10, 14, 8, 17, 29 with 17 (a tile
# of exactly 160 KB at order 4), 2 x 23
@pytest.mark.parametrize("sx,syz,order,n", [(30, 30, 6, 1500), (30, 60, 6, 40), (24, 36, 5, 2000),
                                            (18, 54, 8, 700), (26, 26, 4, 3000), (22, 44, 7, 1),
                                            (32, 16, 3, 2500), (50, 20, 5, 900),
                                            (42, 28, 6, 1100), (8, 40, 8, 300), (34, 34, 4, 600),
                                            (46, 8, 4, 500), (120, 12, 6, 2500)])
@pytest.mark.parametrize("prec,ftol", [("fp64", 1e-10), ("mixed", 1e-5)])
def test_spme_over_bricks(sx, syz, order, n, prec, ftol):
    mesh = np.array([sx, syz, syz])
    box = 1.5 * mesh
    rng = np.random.default_rng(sx * syz + order)
    m = np.maximum((box / 1.4).astype(int), 1)
    # half of the particles in one eighth of the box
    half = np.minimum(m // 2 + 1, m)
    crowd = rng.choice(half.prod(), n // 2, replace=False) if n > 1 else np.zeros(0, int)
    c = np.stack([crowd // (half[1] * half[2]), crowd // half[2] % half[1], crowd % half[2]], 1)
    used = np.zeros(m.prod(), bool)
    used[(c[:, 0] * m[1] + c[:, 1]) * m[2] + c[:, 2]] = True
    free = rng.choice(np.flatnonzero(~used), n - n // 2, replace=False)
    site = np.concatenate([c, np.stack([free // (m[1] * m[2]), free // m[2] % m[1],
                                        free % m[2]], 1)])
    ro = (site + 0.5) * (box / m) - box / 2 + rng.uniform(-0.3, 0.3, (n, 3))
    types = (1 + np.arange(n) % 2).astype(np.int32)
    zat = np.array([1.0, -1.0])
    # no pair within the tables' 0.5 A: the reciprocal part alone
    tab = E.build_tables(zat, np.array([0.3, 0.3]), np.array([1.0, 1.0]), rcut=0.5,
                         epsi_four_pi=EFP, alpha=0.4)
    eng = E.ForceEngine(n, prec)
    eng.set_box(box)
    eng.set_particles(types, zat[types - 1], np.ones(2))
    eng.set_tables(tab, 0.5)
    eng.set_ewald("spm", 0.4, order, mesh, 0, False, False, EFP)
    eng.set_neighbor("vlist", 1.0, 0)
    eng.upload_positions(ro)
    f, en = eng.utotal()
    eng.close()
    orc = O.Oracle(box, types, zat[types - 1], O.Tables(tab.ubuf, tab.iubuflow, tab.nugrid,
                   tab.r2umin, None), 0.5, ewald="spm", alpha=0.4, epsi_four_pi=EFP,
                   order=order, mesh=tuple(int(v) for v in mesh), drnlist=1.0,
                   maxnneigh=max(n, 2))
    orc.set_list(ro)
    fo, eo = orc.utotal(ro)
    if n > 1:
        assert rel_rms(f, fo) <= ftol
    # the scale of the mesh sum (u%rec is that minus the self term)
    mesh_sum = eo["rec"] + EFP * 0.4 / np.sqrt(np.pi) * n
    assert abs(en.rec - eo["rec"]) <= (1e-11 if prec == "fp64" else 1e-6) * mesh_sum
