"""Banded kernel, lattices that do not fill its 64 S sites, with parameters that differ only
in the energies: the padding sites never reach a real one.  Far from resonance (detuning
5.66) a site with the run's drive and interaction but no detuning overflows within the
2000 steps of the launch, so padding stepped that way would put 0 times infinity into the
first and last sites.  The drive of one site moved by 2^-50 of itself is the same number in
FP32 and takes the form with all parameters per site, whose padding has neither drift nor
drive: both forms are the same bit for bit, at either batch size."""
import numpy as np
import pytest

from pincosimulator_amd import Engine, System
from test_gpu_band import matrix_spec

pytestmark = pytest.mark.gpu


def open_band(n, w):
    C = np.zeros((n, n))
    for d in range(1, w + 1):
        for i in range(n - d):
            C[i, i + d] = C[i + d, i] = 0.2
    return C


def open_lieb(cells):
    n = 3 * cells
    C = np.zeros((n, n))
    for a in range(0, n, 3):
        for i, j in ((a, a + 1), (a + 1, a + 2), (a + 2, a + 4)):
            if j < n:
                C[i, j] = C[j, i] = 0.2
    return C


@pytest.mark.parametrize("C", [open_lieb(24), open_band(127, 1), open_band(130, 1), open_band(200, 2), open_band(259, 3),
                               open_lieb(87), open_lieb(127), open_band(510, 2)], ids=lambda c: str(c.shape[0]))
@pytest.mark.parametrize("n_traj", [64, 2500])
def test_padding_reaches_no_site(C, n_traj):
    n = C.shape[0]
    spec = matrix_spec(C, U=3.0, F=0.6, detuning=5.66, omega=0.0, dt=0.005, frame_steps=4000, t_end=10.0)
    ids = np.arange(n_traj, dtype=np.uint64)
    out = []
    for f in (np.full(n, 0.6), np.where(np.arange(n) == n // 2, 0.6 * (1 + 2.0 ** -50), 0.6)):
        print(f"band {n} sites, {n_traj} trajectories", flush=True)
        eng = Engine(System(**dict(spec, F=f)), precision=32, kernel="band")
        out.append(eng.run(ids, final=True).beta_final)
        eng.close()
    stays = np.isfinite(out[1]).all(axis=1)  # noise takes a real site over the same edge in a few trajectories
    assert np.mean(stays) > 0.25
    np.testing.assert_array_equal(out[0][stays], out[1][stays])
