"""Monte Carlo moves over the sizes where the reciprocal pass changes its
form: one moved particle, a full and a partial chunk of eight, the most that
the kernel arguments hold and one more, over meshes of few long and many
short rows and one of more tiles than blocks; trials, accepts and trials
from the kept spectrum against the oracle's reciprocal energies."""
import numpy as np
import pytest

import oracle as O
from test_gpu_fft_lengths import EFP, setup

pytestmark = pytest.mark.gpu

ALPHA, ORDER, N = 0.45, 4, 80


# FP64: summation order against the mesh sum; mixed: FP32 spreading and
# transforms (two accepted changes add in FP64)
@pytest.mark.parametrize("prec,tol", [("fp64", 1e-11), ("mixed", 1e-6)])
@pytest.mark.parametrize("mesh", [(10, 16), (180, 20), (20, 32), (144, 144)],
                         ids=lambda m: "x".join(map(str, m)))
def test_mc_moves_over_sizes(mesh, prec, tol):
    eng, _, ro, box = setup(mesh, N, prec)
    az = np.where(np.arange(N) % 2 == 0, 1.0, -1.0)
    sp = O.SpmeSetup(box, ALPHA, ORDER, (mesh[0], mesh[1], mesh[1]))
    energy = lambda r: EFP * O.spme_rec(sp, r, az, EFP)[1]
    rng = np.random.default_rng(mesh[0])
    u = energy(ro)
    bound = tol * abs(u)
    eng.build_list()
    for it, natm in enumerate((1, 8, 9, 64, 65)):
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
