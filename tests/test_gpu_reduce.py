"""The fold of the partial rows into a frame's sums, at slot counts around its
16 groups and 16 loads in flight, on lattices whose output count leaves a
remainder: equal to the sums over the stored frames, taken in extended
precision (numpy's |z|^2 in FP64 is itself several ulp off).  A term |z|^4 is
rounded by at most 5 2^-53 and B terms of one sign pattern add at most B 2^-53
each way, so the sums are within 2 (B + 2) 2^-53 of the sum of magnitudes."""
import numpy as np
import pytest

from pincosimulator_amd import Engine, System

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("precision,kernel", [(64, "generic"), (32, "auto")])
@pytest.mark.parametrize("nx,ny", [(1, 5), (6, 11)])
@pytest.mark.parametrize("n_traj", [1, 15, 17, 255, 257, 1025])
def test_frame_sums_fold(precision, kernel, nx, ny, n_traj):
    print(f"fold FP{precision} {nx}x{ny} {n_traj}", flush=True)
    s = System(nx=nx, ny=ny, dt=0.004, gamma=1.0, J=1.0, omega=0.5, U=0.06, F=1.1, beta_init=0.0, beta_sigma=0.5,
               frame_steps=3, seed=41, t_start=0.0, t_end=0.025)
    eng = Engine(s, precision=precision, kernel=kernel)
    for _ in range(2):  # the second batch finds the rows as the first left them
        res = eng.run(np.arange(n_traj), traj=True)
    eng.close()
    z = res.traj.astype(np.clongdouble)
    q = z.real ** 2 + z.imag ** 2
    ref = {"sum_n": q.sum(axis=0), "sum_n2": (q * q).sum(axis=0), "sum_beta": z.sum(axis=0)}
    mag = {"sum_n": ref["sum_n"], "sum_n2": ref["sum_n2"], "sum_beta": np.sqrt(q).sum(axis=0)}
    for k, m in mag.items():
        assert np.all(np.abs(getattr(res, k) - ref[k]) <= 2 * (n_traj + 2) * 2.0 ** -53 * m), k
