"""Adjoint and force matching with spline tables whose sums take up to a
block's LDS (160 KB): eight types of about 64 KB (7,884 and 7,920
coefficients), 20,196 that fit the adjoint and 20,454 and 20,448 that fit
force matching beside the kernels' other sums, against autograd of the pair
model over all pairs in FP64; larger tables are refused, by the gradients
alone."""
import numpy as np
import pytest
import torch

from molsim_amd import engine as E
from test_gpu_adjoint_sizes import EFP, R_LO, RC, check_force_matching, model

pytestmark = pytest.mark.gpu


def system(npt, nknot, prec):
    n, L = 120, 40.0
    rng = np.random.default_rng(nknot)
    site = rng.choice(6 ** 3, n, replace=False)
    x = np.stack([site // 36, site // 6 % 6, site % 6], 1) * 3.0
    x = x - x.mean(0) + rng.uniform(-0.3, 0.3, (n, 3))
    types = (1 + np.arange(n) % npt).astype(np.int32)
    zat = np.where(np.arange(npt) % 2 == 0, 1.0, -1.0)
    sig, eps = 2.8 + 0.05 * np.arange(npt), 0.7 + 0.1 * np.arange(npt)
    c = 0.1 * rng.standard_normal((npt * (npt + 1) // 2, nknot))
    tab = E.build_tables(zat, sig, eps, rcut=RC, epsi_four_pi=EFP, lewald=False)
    eng = E.ForceEngine(n, prec)
    eng.set_box(L)
    eng.set_particles(types, zat[types - 1], np.ones(npt))
    eng.set_tables(tab, RC)
    eng.set_ewald("none", 0.0, 0, (0, 0, 0), 1, False, False, EFP)
    eng.set_neighbor("vlist", 2.0, n)
    eng.set_pair_params(zat, sig, eps, rcut=RC, epsi_four_pi=EFP, lewald=False)
    eng.set_knots(R_LO, RC, c)
    eng.upload_positions(x)
    return eng, x, types, L, zat, sig, eps, c, rng


def reference(x, types, L, zat, sig, eps, c):
    t = [torch.tensor(v, dtype=torch.float64, requires_grad=True) for v in
         (x, zat, sig, eps, c)]
    e = model(t[0], torch.tensor(types - 1).long(), L, *t[1:])
    return t, float(e.detach()), torch.autograd.grad(e, t, create_graph=True)


# the bounds of test_gpu_adjoint_sizes.py; force matching in FP64 as there
@pytest.mark.parametrize("npt,nknot", [(8, 219), (8, 220), (8, 561)])
@pytest.mark.parametrize("prec,tol", [("fp64", 1e-10), ("mixed", 2e-5)])
def test_adjoint_of_large_knot_tables(npt, nknot, prec, tol):
    eng, *s, rng = system(npt, nknot, prec)
    t, e, g = reference(*s)
    got = eng.adjoint()
    assert abs(got["E"] - e) <= tol * max(abs(e), 1.0)
    for name, k in (("dzat", 1), ("dsigat", 2), ("depsat", 3), ("dknot", 4)):
        want = g[k].detach().numpy()
        assert np.abs(got[name] - want).max() <= tol * (np.abs(want).max() + 1), name
    eng.close()


@pytest.mark.parametrize("npt,nknot", [(8, 220), (6, 974), (8, 568)])
def test_force_matching_of_large_knot_tables(npt, nknot):
    eng, *s, rng = system(npt, nknot, "fp64")
    t, _, g = reference(*s)
    check_force_matching(eng, t, g, s[0], 1, rng, 1e-9)
    eng.close()


@pytest.mark.parametrize("prec", ["fp64", "mixed"])
def test_tables_beyond_a_block_are_refused(prec):
    eng, x = system(8, 1024, prec)[:2]
    f, _ = eng.utotal()
    assert np.isfinite(f).all()
    eng.fm_set_frames(x[None], np.zeros((1,) + x.shape))
    for call in (eng.adjoint, eng.fm_loss_grad):
        with pytest.raises(E.MfeError, match="LDS"):
            call()
    f2 = eng.model_forces()
    assert np.isfinite(f2).all()
    eng.close()
