"""The list build with each number of lanes per particle (1, 4, 16) and the
pair kernels with each (1 to 64), the counts worked out here from the sizes
as the engine does, so that no branch goes untested when a threshold moves:
lists against all pairs, pair forces and energies against the oracle."""
import numpy as np
import pytest
from scipy.spatial import cKDTree

from molsim_amd import engine as E
import test_gpu_pair_lanes as pair_lanes

pytestmark = pytest.mark.gpu

SKIN = 2.0


def cells(box, rc):
    n = np.floor(np.broadcast_to(box, 3) / (rc + SKIN)).astype(int)
    return np.where(n < 3, 1, n)


def list_lanes(box, n, rc):
    row = 3.0 * n / cells(box, rc).prod()
    if row < 8.0:
        return 1
    return 16 if row >= 20.0 and n <= 32768 else (4 if n <= 262144 else 1)


def pair_lanes_of(L, n, rc, prec):
    m = 4.0 / 3.0 * np.pi * (rc + SKIN) ** 3 * n / L ** 3
    lanes = 4
    if prec == "mixed" and cells(L, rc).min() >= 3:
        lanes = 1 if m <= 12.0 else (2 if m <= 48.0 else 4)
    while lanes < 64 and 2 * lanes * n <= 131072 and m >= 8 * lanes:
        lanes *= 2
    return lanes


LISTS = [((70.0, 70.0, 70.0), 300, 10.0, 1), ((75.0, 75.0, 75.0), 600, 13.0, 4),
         ((90.0, 75.0, 77.0), 901, 13.0, 4), ((190.0, 190.0, 190.0), 33000, 9.0, 4),
         ((66.0, 60.0, 84.0), 900, 18.0, 16)]
PAIRS = [(60.0, 200, 10.0, 2, 1, 4), (60.0, 420, 10.0, 2, 2, 4), (60.0, 420, 10.0, 5, 2, 4),
         (200.0, 20000, 12.0, 3, 4, 4), (60.0, 1100, 10.0, 3, 8, 8), (66.0, 2100, 12.0, 4, 16, 16),
         (70.0, 1400, 18.0, 2, 32, 32), (70.0, 1700, 18.0, 5, 32, 32), (64.0, 2048, 18.0, 3, 64, 64)]


def test_every_lane_count_has_a_case():
    assert {list_lanes(*c[:3]) for c in LISTS} == {1, 4, 16}
    assert all(list_lanes(*c[:3]) == c[3] for c in LISTS)
    for k, prec in ((4, "mixed"), (5, "fp64")):
        assert all(pair_lanes_of(*c[:3], prec) == c[k] for c in PAIRS)
    assert {c[4] for c in PAIRS} == {1, 2, 4, 8, 16, 32, 64}
    assert {c[5] for c in PAIRS} == {4, 8, 16, 32, 64}


def pairs_within(ro, box, rs):
    """SetVListMD's membership test on the pairs a tree finds within a
    little more than rs: one shift per axis, squares summed left to right."""
    tree = cKDTree(np.mod(ro + box / 2, box) % box, boxsize=box)
    ij = tree.query_pairs(rs * (1.0 + 1e-9), output_type="ndarray")
    d = ro[ij[:, 0]] - ro[ij[:, 1]]
    d = np.where(np.abs(d) > box / 2, d - np.copysign(box, d), d)
    r2 = (d[:, 0] * d[:, 0] + d[:, 1] * d[:, 1]) + d[:, 2] * d[:, 2]
    ij = np.sort(ij[r2 < rs * rs], 1)
    return ij[np.lexsort((ij[:, 1], ij[:, 0]))]


@pytest.mark.parametrize("box,n,rc,lanes", LISTS)
@pytest.mark.parametrize("prec", ["mixed", "fp64"])
def test_list_of_every_lane_count(box, n, rc, lanes, prec):
    box = np.array(box)
    rng = np.random.default_rng(n)
    ro = rng.uniform(-0.5, 0.5, (n, 3)) * box
    # a tenth of the particles crowded into a corner
    k = n // 10
    ro[:k] = -box / 2 + rng.uniform(0.0, 0.3, (k, 3)) * box
    types = (1 + np.arange(n) % 2).astype(np.int32)
    zat = np.array([1.0, -1.0])
    tab = E.build_tables(zat, np.array([0.1, 0.1]), np.array([0.1, 0.1]), rcut=rc,
                         epsi_four_pi=E.epsi0_four_pi() / 78.4, alpha=3.0 / rc)
    eng = E.ForceEngine(n, prec)
    eng.set_box(box)
    eng.set_particles(types, zat[types - 1], np.ones(2))
    eng.set_tables(tab, rc)
    most = min(n - 1, 400)
    eng.set_neighbor("vlist", SKIN, most)
    eng.upload_positions(ro)
    # the explicit build, then the gated one after a move that fires the
    # skin test
    for step in range(2):
        if step:
            ro = np.clip(ro + rng.uniform(-3.0, 3.0, ro.shape), -box / 2, box / 2)
            eng.upload_positions(ro)
        else:
            eng.build_list()
        nn, jl = eng.get_pairs(most)
        i = np.repeat(np.arange(n), nn)
        j = np.concatenate([jl[a, :nn[a]] for a in range(n)]) - 1
        got = np.sort(np.stack([i, j], 1), 1)
        got = got[np.lexsort((got[:, 1], got[:, 0]))]
        assert np.array_equal(got, pairs_within(ro, box, rc + SKIN))
    eng.close()


@pytest.mark.parametrize("L,n,rc,ntype,mixed,fp64", PAIRS)
@pytest.mark.parametrize("prec", ["mixed", "fp64"])
def test_pairs_of_every_lane_count(L, n, rc, ntype, mixed, fp64, prec):
    pair_lanes.test_pair_lanes_vs_oracle(L, n, rc, "vlist", ntype, prec)
