"""Mixed precision with an axis of 1024 points (three radices, the fewest
columns and rows per block): forces, energies, virial and a Monte Carlo
change against the oracle."""
import numpy as np
import pytest

from test_gpu_fft_lengths import EFP, setup

from helpers import rel_rms

pytestmark = pytest.mark.gpu


# the energy bounds of test_gpu_fft_lengths.py; forces: FP32 amplitudes of a
# sum along 1024 points (its bound of 1e-5 is for up to 512 points), while a
# wrong index gives errors of order one
@pytest.mark.parametrize("mesh", [(1024, 16), (8, 1024), (1024, 32)],
                         ids=lambda m: "x".join(map(str, m)))
def test_mixed_spme_on_long_axes(mesh):
    eng, orc, ro, box = setup(mesh, 60, "mixed")
    f, en = eng.utotal()
    orc.set_list(ro)
    fo, eo = orc.utotal(ro)
    assert rel_rms(f, fo) <= 5e-5
    mesh_sum = eo["rec"] + EFP * 0.45 / np.sqrt(np.pi) * ro.shape[0]
    assert abs(en.rec - eo["rec"]) <= 1e-6 * mesh_sum
    assert abs(en.virial - eo["virial"]) <= 1e-5 * mesh_sum
    new = ro.copy()
    new[7] = np.clip(ro[7] + np.array([0.4, -0.3, 0.2]), -box / 2, box / 2)
    du = eng.mc_delta_rec([8], new[7:8])
    _, en_new = orc.utotal(new)
    assert abs(du - (en_new["rec"] - eo["rec"])) <= 1e-6 * mesh_sum
    eng.close()
