"""The step kernels that take trajectories from a queue in long launches and a fixed share
per workgroup in short ones: one launch of all steps and launches of one step give the
same states bit for bit, with more trajectories than workgroups (both ways) and with
fewer; two trajectories against the FP64 oracle."""
import numpy as np
import pytest

import oracle
from helpers import FP32_BAR, c2_spec, oracle_params, rel_err, system
from pincosimulator_amd import Engine

pytestmark = pytest.mark.gpu

CASES = [(64, 64, 32, {}, 1100), (63, 63, 32, {}, 1100), (17, 21, 32, {}, 4200), (5, 13, 32, {}, 9000),
         (32, 32, 32, dict(F=1.0 + 0.2j * np.cos(np.arange(1024))), 1300), (64, 64, 64, {}, 700), (40, 41, 64, {}, 1100),
         (64, 64, 32, {}, 100)]


@pytest.mark.parametrize("nx,ny,precision,form,n_traj", CASES, ids=[f"{c[0]}x{c[1]}-{c[2]}-{c[4]}" for c in CASES])
def test_queue_and_shares_agree(nx, ny, precision, form, n_traj):
    steps = (20000 + nx * ny - 1) // (nx * ny) + 1  # of one launch; the queue from 20000 site-steps on, FP64 8192
    ids = np.arange(n_traj, dtype=np.uint64) * 3 + 1
    out = []
    for frame_steps in (steps, 1):
        print(f"{nx}x{ny}, FP{precision}, {n_traj} trajectories, {frame_steps} steps a launch", flush=True)
        spec = c2_spec(**dict(dict(nx=nx, ny=ny, dt=0.005, J=0.7, U=0.08, t_end=0.005 * (steps + 0.25),
                                   frame_steps=frame_steps), **form))
        eng = Engine(system(spec), precision=precision)
        res = eng.run(ids, final=True)
        eng.close()
        out.append(res.beta_final)
        assert res.n_steps == steps
    np.testing.assert_array_equal(out[0], out[1])
    for j in (0, n_traj - 1):
        assert rel_err(out[0][j], oracle.run_trajectory(oracle_params(spec), int(ids[j]))[1]) < (FP32_BAR if precision == 32
                                                                                               else 1e-9)
