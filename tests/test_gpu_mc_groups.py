"""Pair changes of Monte Carlo moves of neighbours: groups of particles
around a point, so that most of a moved particle's partners within the
cut-off move too, and pairs between them count once, against the oracle's
two-body energy of both configurations (FP64 on both engine paths: the
bound of the other pair changes, 1e-10 of |u_twob|)."""
import numpy as np
import pytest

from molsim_amd import engine as E
from molsim_amd import systems as S
from helpers import efp, oracle_for

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("natm", [2, 8, 64, 65])
@pytest.mark.parametrize("nlist", ["vlist", "cell"])
@pytest.mark.parametrize("prec", ["fp64", "mixed"])
def test_mc_delta_pair_of_neighbours(natm, nlist, prec):
    s = S.c2()
    tab = E.build_tables(s.zat, s.sigat, s.epsat, rcut=s.rcut, epsi_four_pi=efp(),
                         alpha=s.alpha)
    eng = S.configure(s, prec, tables=tab, nlist=nlist)
    eng.build_list()
    orc = oracle_for(s, tab, nlist=nlist)
    orc.set_list(s.ro)
    u0 = orc.utotal(s.ro)[1]["twob0"]
    d = s.ro - s.ro[7]
    d -= s.boxlen * np.round(d / s.boxlen)
    ia = np.argsort((d * d).sum(1))[:natm]
    rng = np.random.default_rng(natm)
    rtm = s.ro[ia] + rng.uniform(-0.1, 0.1, (natm, 3))
    rtm -= s.boxlen * np.round(rtm / s.boxlen)
    du, ov = eng.mc_delta_pair(ia + 1, rtm)
    ro1 = s.ro.copy()
    ro1[ia] = rtm
    if nlist == "cell":
        orc.set_list(ro1)
    u1 = orc.utotal(ro1)[1]["twob0"]
    print(f"du {du:.10e} oracle {u1 - u0:.10e}", flush=True)
    assert not ov and du != 0.0
    assert abs(du - (u1 - u0)) <= 1e-10 * abs(u0)
    # onto a particle that stays
    rtm[0] = s.ro[np.argsort((d * d).sum(1))[natm]] + 0.1
    assert eng.mc_delta_pair(ia + 1, rtm) == (0.0, True)
    eng.close()
