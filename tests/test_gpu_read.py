"""FP32 trajectories read back in one piece and in chunks (1 MiB and more, 512 KiB a
chunk, four readers): sizes around the limit, whole and partial last chunks, fewer
and more chunks than readers; every state against the frame's own sums and means."""
import numpy as np
import pytest

from helpers import c2_spec, rel_err, system
from pincosimulator_amd import Engine

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("n_traj", [1, 341, 342, 512, 513, 700, 2731, 8193])
def test_fp32_states_read_back(n_traj):
    spec = c2_spec(nx=8, ny=16, dt=0.01, frame_steps=2, t_end=0.0425)  # 1 KiB a state, three frames
    print(f"read {n_traj} trajectories", flush=True)
    eng = Engine(system(spec), precision=32)
    for _ in range(2):
        res = eng.run(np.arange(n_traj, dtype=np.uint64), traj=True, final=True)
        assert res.traj.shape == (n_traj, 3, 128)
        n = np.abs(res.traj) ** 2
        assert rel_err(res.traj_m2, n.mean(axis=2)) < 1e-12
        assert rel_err(res.sum_beta, res.traj.sum(axis=0)) < 1e-12
        np.testing.assert_array_equal(res.beta_final, res.traj[:, -1])
    eng.close()
