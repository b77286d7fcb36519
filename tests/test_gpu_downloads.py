"""Downloads at the edges of the pinned ring: one slot's worth, whole and
partial slots, more chunks than slots, of one and of three arrays, against
the values that were uploaded (bitwise)."""
import numpy as np
import pytest

from molsim_amd import engine as E

pytestmark = pytest.mark.gpu

MB = 1 << 20


# particles whose positions take about that many bytes: below the ring's
# least, at it, at the change of the slot, and beyond 16 slots
@pytest.mark.parametrize("n", [1, 43690, 87381, 87382, 233017, 699051, 1500001])
def test_state_comes_back_as_uploaded(n):
    rng = np.random.default_rng(n)
    ro = rng.uniform(-100.0, 100.0, (n, 3))
    rod, rodd = rng.standard_normal((2, n, 3))
    with E.ForceEngine(n, "fp64") as eng:
        eng.set_box([200.0] * 3)
        eng.set_particles(np.ones(n, np.int32), np.zeros(n), np.ones(1))
        eng.upload_positions(ro)
        eng.upload_velocities(rod, rodd)
        for _ in range(2):
            for got, want in zip(eng.download_state(), (ro, rod, rodd)):
                assert np.array_equal(got, want)
        # one coordinate outside, at the start, in the middle or at the end,
        # is refused, as is NaN
        for k in (0, 3 * (n // 2) + 1, 3 * n - 1):
            for bad in (100.0 + 1e-9, -100.1, np.nan):
                x = ro.copy().reshape(-1)
                x[k] = bad
                with pytest.raises(E.MfeError):
                    eng.upload_positions(x)
        assert np.array_equal(eng.download_state()[0], ro)
