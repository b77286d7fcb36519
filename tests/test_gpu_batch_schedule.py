"""The BD schedule a batch takes by itself, and the per-stage launches of a
batch that fills the chip (the pair launch beside the SPME stages) against
each engine alone."""
import numpy as np
import pytest

from molsim_amd import engine as E
from molsim_amd import systems as S

pytestmark = pytest.mark.gpu


def replica(r, tab):
    s = S.c4_replica(r, mesh=36, order=4)
    n = 2 * (20 + 7 * r % 90)
    keep = np.concatenate([np.arange(n // 2), s.np // 2 + np.arange(n // 2)])
    s.ro, s.rod, s.iptpn = s.ro[keep], s.rod[keep], s.iptpn[keep]
    s.rcut, s.alpha = 12.0, 0.25
    if tab is None:
        tab = E.build_tables(s.zat, s.sigat, s.epsat, rcut=12.0,
                             epsi_four_pi=E.epsi0_four_pi() / 78.4, alpha=0.25)
    e = S.configure(s, "mixed", tables=tab, maxnneigh=s.np - 1)
    e.set_bd([0.002, 0.002], [0.05, 0.05], 50 + r)
    return e, tab


@pytest.mark.parametrize("nrep", [1, 3, 100])
def test_small_batches_replay_the_per_stage_graph(nrep):
    tab, engs, alone = None, [], []
    for r in range(nrep):
        e, tab = replica(r, tab)
        engs.append(e)
    pick = sorted({0, nrep // 2, nrep - 1})
    for r in pick:
        e, _ = replica(r, tab)
        e.utotal()
        e.step_bd(nsteps=9)
        e.step_bd(nsteps=4)
        alone.append((e.download_state()[0], e.download_forces(), e.energy().tot))
        e.close()
    with E.Batch(engs) as b:
        b.compute()
        assert not b.uses_persistent()
        b.set_persistent(True)
        assert b.uses_persistent()
        b.set_persistent(False)
        assert not b.uses_persistent()
        b.step_bd(9)
        b.step_bd(4)
        en = b.energies()
        for r, (ro, f, tot) in zip(pick, alone):
            assert np.array_equal(engs[r].download_state()[0], ro)
            assert np.array_equal(engs[r].download_forces(), f)
            assert abs(en[r].tot - tot) <= 1e-12 * max(abs(tot), 1.0)
    for e in engs:
        e.close()
