"""Monte Carlo moves around the number of particles from which the factors
come from a table, with partial chunks of it, over a mesh of many short
rows, a large one (four points per thread) and one whose x factors leave
room for a single particle: trials, accepts and trials from the kept
spectrum against the oracle's reciprocal energies."""
import numpy as np
import pytest

import oracle as O
from test_gpu_fft_lengths import EFP, setup

pytestmark = pytest.mark.gpu

ALPHA, ORDER, N = 0.45, 4, 80


# the bounds of test_gpu_mc_sizes.py
@pytest.mark.parametrize("mesh,prec,tol", [((10, 16), "fp64", 1e-11), ((10, 16), "mixed", 1e-6),
                                           ((144, 144), "fp64", 1e-11),
                                           ((144, 144), "mixed", 1e-6),
                                           ((1024, 16), "fp64", 1e-11)])
def test_mc_moves_from_the_factor_table(mesh, prec, tol):
    eng, _, ro, box = setup(mesh, N, prec)
    az = np.where(np.arange(N) % 2 == 0, 1.0, -1.0)
    sp = O.SpmeSetup(box, ALPHA, ORDER, (mesh[0], mesh[1], mesh[1]))
    energy = lambda r: EFP * O.spme_rec(sp, r, az, EFP)[1]
    rng = np.random.default_rng(mesh[0])
    u = energy(ro)
    bound = tol * abs(u)
    eng.build_list()
    for it, natm in enumerate((2, 3, 23, 2, 70, 3)):
        ia = rng.choice(N, natm, replace=False)
        new = ro.copy()
        new[ia] = np.clip(ro[ia] + rng.uniform(-0.2, 0.2, (natm, 3)), -box / 2, box / 2)
        du = eng.mc_delta_rec(ia + 1, new[ia], reuse_current=it > 0)
        u_new = energy(new)
        print(f"{natm}: du {du:.10e} oracle {u_new - u:.10e}", flush=True)
        assert abs(du - (u_new - u)) <= bound
        eng.mc_accept(ia + 1, new[ia])
        ro, u = new, u_new
    assert np.array_equal(eng.download_state()[0].reshape(-1, 3), ro)
    eng.close()
