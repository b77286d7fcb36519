"""List build with 1, 4 and 16 lanes per particle, crowded cells and boxes
that are one cell, against an FP64 brute force over all pairs."""
import numpy as np
import pytest

from molsim_amd import engine as E

pytestmark = pytest.mark.gpu


def brute_pairs(ro, box, rs):
    """SetVListMD's membership test on every pair: one shift per axis and
    the three squares summed left to right."""
    out = set()
    n = ro.shape[0]
    for i in range(n - 1):
        d = ro[i] - ro[i + 1:]
        d = np.where(np.abs(d) > box / 2, d - np.copysign(box, d), d)
        r2 = (d[:, 0] * d[:, 0] + d[:, 1] * d[:, 1]) + d[:, 2] * d[:, 2]
        out.update((i, i + 1 + int(j)) for j in np.flatnonzero(r2 < rs * rs))
    return out


# box, particles, cut-off: rows of cells with fewer than 8 members (one
# lane), 8 to 48 (4 lanes), more (16 lanes), one cell, one cell on two axes
@pytest.mark.parametrize("prec", ["mixed", "fp64"])
@pytest.mark.parametrize("box,n,rc", [((70.0, 70.0, 70.0), 300, 10.0),
                                      ((90.0, 78.0, 120.0), 3001, 13.0),
                                      ((66.0, 60.0, 84.0), 2500, 18.0),
                                      ((50.0, 50.0, 50.0), 1000, 15.0),
                                      ((40.0, 40.0, 140.0), 777, 15.0),
                                      ((60.0, 60.0, 60.0), 2, 12.0)])
def test_list_equals_brute_force(box, n, rc, prec):
    box = np.array(box)
    rng = np.random.default_rng(n)
    # a third of the particles crowded into a corner
    ro = rng.uniform(-0.5, 0.5, (n, 3)) * box
    ro[: n // 3] = -box / 2 + rng.uniform(0.0, 0.3, (n // 3, 3)) * box
    types = (1 + np.arange(n) % 2).astype(np.int32)
    zat = np.array([1.0, -1.0])
    tab = E.build_tables(zat, np.array([0.1, 0.1]), np.array([0.1, 0.1]), rcut=rc,
                         epsi_four_pi=E.epsi0_four_pi() / 78.4, alpha=3.0 / rc)
    eng = E.ForceEngine(n, prec)
    eng.set_box(box)
    eng.set_particles(types, zat[types - 1], np.ones(2))
    eng.set_tables(tab, rc)
    eng.set_neighbor("vlist", 2.0, n)
    eng.upload_positions(ro)
    want = brute_pairs(ro, box, rc + 2.0)
    # the explicit build, then the gated one after a move that fires the
    # skin test
    for step in range(2):
        if step:
            ro = np.clip(ro + rng.uniform(-3.0, 3.0, ro.shape), -box / 2, box / 2)
            eng.upload_positions(ro)
            want = brute_pairs(ro, box, rc + 2.0)
        else:
            eng.build_list()
        nn, jl = eng.get_pairs(n)
        got = [(min(i, j - 1), max(i, j - 1)) for i in range(n) for j in jl[i, :nn[i]]]
        assert len(got) == len(want)
        assert set(got) == want
    eng.close()
