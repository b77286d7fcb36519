"""The choice of the brick edges where it turns, against the oracle: tiles
near the LDS of a CU (axes of 2 x 31 points beside an axis whose largest
brick would not fit with them) and the particles per brick above which few
bricks are made smaller."""
import numpy as np
import pytest

import oracle as O
from molsim_amd import engine as E
from helpers import rel_rms

pytestmark = pytest.mark.gpu

EFP = E.epsi0_four_pi() / 78.4


def against_oracle(mesh, order, n, prec, ftol):
    """UTotal of n ions on distinct sites without pair forces; the bounds
    are those of the other brick tests."""
    mesh = np.array(mesh)
    box = 1.5 * mesh
    rng = np.random.default_rng(int(mesh[0] * mesh[1]) + order)
    m = np.maximum((box / 1.4).astype(int), 1)
    site = rng.choice(m.prod(), n, replace=False)
    site = np.stack([site // (m[1] * m[2]), site // m[2] % m[1], site % m[2]], 1)
    ro = (site + 0.5) * (box / m) - box / 2 + rng.uniform(-0.3, 0.3, (n, 3))
    types = (1 + np.arange(n) % 2).astype(np.int32)
    zat = np.array([1.0, -1.0])
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
    # positions that move with the list kept: nothing of the set-up above is
    # reported by a later call
    eng.upload_positions(np.clip(ro + 0.01, -box / 2, box / 2))
    eng.upload_positions(ro)
    assert rel_rms(eng.utotal()[0], f) <= ftol
    eng.close()
    orc = O.Oracle(box, types, zat[types - 1], O.Tables(tab.ubuf, tab.iubuflow, tab.nugrid,
                   tab.r2umin, None), 0.5, ewald="spm", alpha=0.4, epsi_four_pi=EFP,
                   order=order, mesh=tuple(int(v) for v in mesh), drnlist=1.0,
                   maxnneigh=max(n, 2))
    orc.set_list(ro)
    fo, eo = orc.utotal(ro)
    assert rel_rms(f, fo) <= ftol
    # the scale of the mesh sum (u%rec is that minus the self term)
    mesh_sum = eo["rec"] + EFP * 0.4 / np.sqrt(np.pi) * n
    assert abs(en.rec - eo["rec"]) <= (1e-11 if prec == "fp64" else 1e-6) * mesh_sum


# 62 = 2 x 31 and 58 = 2 x 29 have no divisor from 8 to 16: their bricks leave
# room for an edge of 8 (24) or 10 (30) on the third axis, not for 12 or 15
@pytest.mark.parametrize("mesh,order,n", [((24, 62, 62), 6, 900), ((30, 62, 62), 6, 700),
                                          ((24, 58, 58), 8, 800)])
@pytest.mark.parametrize("prec,ftol", [("fp64", 1e-10), ("mixed", 1e-5)])
def test_small_edge_beside_large_ones(mesh, order, n, prec, ftol):
    against_oracle(mesh, order, n, prec, ftol)


# bricks of 17 x 29 x 29 at order 4: a tile of exactly 160 KB, which has no room
# for an odd plane nor, in FP64, for a launch's own LDS beside it
@pytest.mark.parametrize("prec,ftol", [("fp64", 1e-10), ("mixed", 1e-5)])
def test_tile_of_a_whole_lds(prec, ftol):
    against_oracle((34, 58, 58), 4, 600, prec, ftol)


# 24^3 at order 6 is eight bricks of edge 12 up to 2^16 (FP64) or 2^17 (mixed)
# stencil points per brick, 2427 and 4854 particles, then 27 of edge 8
@pytest.mark.parametrize("n", [2427, 2428, 4854, 4855])
@pytest.mark.parametrize("prec,ftol", [("fp64", 1e-10), ("mixed", 1e-5)])
def test_few_crowded_bricks(n, prec, ftol):
    against_oracle((24, 24, 24), 6, n, prec, ftol)
