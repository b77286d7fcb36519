"""Per-stage batch steps give every replica the energies that its engine
gives alone, bit for bit, as positions and forces."""
import numpy as np
import pytest

from molsim_amd import engine as E
from test_gpu_batch_schedule import replica

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("kind", ["bd", "md"])
@pytest.mark.parametrize("nrep", [2, 100])
def test_energies_equal_the_engine_alone(nrep, kind):
    tab, engs, alone = None, [], []
    for r in range(nrep):
        e, tab = replica(r, tab)
        engs.append(e)
    step = (lambda x, k: x.step_md(k, 0.001)) if kind == "md" else (
        lambda x, k: x.step_bd(nsteps=k) if isinstance(x, E.ForceEngine) else x.step_bd(k))
    pick = sorted({0, nrep // 2, nrep - 1})
    for r in pick:
        e, _ = replica(r, tab)
        e.utotal()
        step(e, 9)
        step(e, 4)
        alone.append((e.download_forces(), e.energy()))
        e.close()
    with E.Batch(engs) as b:
        b.set_persistent(False)
        b.compute()
        step(b, 9)
        step(b, 4)
        en = b.energies()
        for r, (f, one) in zip(pick, alone):
            assert np.array_equal(engs[r].download_forces(), f)
            assert (en[r].tot, en[r].rec, en[r].virial) == (one.tot, one.rec, one.virial)
            assert np.array_equal(en[r].twob, one.twob)
    for e in engs:
        e.close()
