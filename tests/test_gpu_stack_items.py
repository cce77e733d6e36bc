"""Items of the stacked step kernel where they can go wrong: one and two pairs per
thread with a last wave partly filled, one trajectory per item and stacked ones
with a short last item, more items than workgroup slots, an odd number of steps
per launch, a complex interaction -- against the FP64 oracle, and the same
trajectory from batches of different sizes (and so different stacking) bit for
bit."""
import numpy as np
import pytest

import oracle
from helpers import FP32_BAR, rel_err, system
from pincosimulator_amd import Engine

pytestmark = pytest.mark.gpu


def spec(nx, ny, **kw):
    s = dict(nx=nx, ny=ny, dt=0.004, gamma=1.0, J=0.9, omega=0.4, U=0.06, F=1.3, beta_init=0.0, beta_sigma=0.5,
             frame_steps=7, seed=99, t_start=0.0, t_end=0.084)
    s.update(kw)
    return s


@pytest.mark.parametrize("nx,ny", [(2, 34), (1, 66), (6, 22), (36, 50), (45, 46), (64, 62), (64, 64), (8, 512), (1, 512)])
@pytest.mark.parametrize("n_traj", [1, 5, 1100])
@pytest.mark.parametrize("U", [0.06, 0.06 + 0.03j])
def test_items_match_oracle(nx, ny, n_traj, U):
    sp = spec(nx, ny, U=U)
    print(f"stack {nx}x{ny} x {n_traj} U={U}", flush=True)
    eng = Engine(system(sp), precision=32, kernel="stack")
    ids = np.arange(n_traj, dtype=np.uint64) * 7 + (1 << 33) - 3000   # ids on both sides of 2^33
    out = eng.run(ids, final=True).beta_final
    p = dict(sp, lattice=oracle.LAT_FFT)
    for j in sorted({0, n_traj // 2, n_traj - 1}):
        assert rel_err(out[j], oracle.run_trajectory(p, int(ids[j]))[1]) < FP32_BAR
    np.testing.assert_array_equal(eng.run(ids[-2:], final=True).beta_final, out[-2:])
    eng.close()
