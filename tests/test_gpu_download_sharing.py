"""The pinned ring that a device's engines share: downloads of engines of
different sizes in turn (the ring grows), from threads at once (one has the
ring, the others the runtime's copy), after an engine is closed and after
all are, against the values that were uploaded (bitwise)."""
import threading

import numpy as np
import pytest

from molsim_amd import engine as E

pytestmark = pytest.mark.gpu


def make(n):
    rng = np.random.default_rng(n)
    state = (rng.uniform(-100.0, 100.0, (n, 3)), *rng.standard_normal((2, n, 3)))
    eng = E.ForceEngine(n, "fp64")
    eng.set_box([200.0] * 3)
    eng.set_particles(np.ones(n, np.int32), np.zeros(n), np.ones(1))
    eng.upload_positions(state[0])
    eng.upload_velocities(*state[1:])
    return eng, state


def same(eng, state):
    return all(np.array_equal(a, b) for a, b in zip(eng.download_state(), state))


def test_engines_share_the_ring():
    pairs = [make(n) for n in (60000, 150001, 300007)]
    for _ in range(2):
        for eng, state in pairs:
            assert same(eng, state)
    bad = []

    def work(eng, state):
        for _ in range(8):
            if not same(eng, state):
                bad.append(state[0].shape)

    threads = [threading.Thread(target=work, args=p) for p in pairs]
    for t in threads:
        t.start()
    for t in threads:
        t.join()
    assert not bad
    pairs[2][0].close()
    for eng, state in pairs[:2]:
        assert same(eng, state)
        eng.close()
    eng, state = make(90001)
    assert same(eng, state)
    eng.close()
