"""Dense couplings of 2 to 512 sites on the matrix-core kernel: sites at the edges of its
row tiles, waves and padded sizes (rows, waves and k blocks past the lattice), 16 and 32
trajectories per workgroup with a last one partly filled; against the FP64 oracle,
and the same trajectories from either batch size bit for bit."""
import numpy as np
import pytest
import torch

import oracle
from helpers import FP32_BAR, rel_err
from pincosimulator_amd import Engine, System

pytestmark = pytest.mark.gpu

SITES = [2, 15, 16, 17, 33, 96, 97, 128, 129, 160, 224, 225, 256, 257, 351, 352, 353, 384, 385, 480, 481, 512]


@pytest.mark.parametrize("n", SITES)
def test_shapes_match_oracle(n):
    rng = np.random.default_rng(n)
    spec = dict(nx=1, ny=n, dt=0.005, gamma=1.0, J=0.0, U=np.linspace(0.05, 0.1, n) + 0.02j,
                F=1.2 * np.exp(1j * rng.uniform(0, 6, n)), omega=0.3 * rng.standard_normal(n), beta_init=0.0,
                beta_sigma=0.5, frame_steps=7, seed=n, t_start=0.0, t_end=0.005 * 10.25, lattice="matrix",
                coupling=rng.uniform(-1.0, 1.0, (n, n)) * (2.0 / np.sqrt(n)), detuning=0.2, onsite="detuning-E")
    ids = np.arange(16 * torch.cuda.get_device_properties(0).multi_processor_count + 21, dtype=np.uint64) * 3 + 1
    print(f"mfma {n} sites", flush=True)
    eng = Engine(System(**spec), precision=32, kernel="mfma")
    res = eng.run(ids, final=True)
    p = dict(spec, lattice=oracle.LAT_DENSE, E=spec["omega"])
    for j in (0, 2000, len(ids) - 1):
        assert rel_err(res.beta_final[j], oracle.run_trajectory(p, int(ids[j]))[1]) < FP32_BAR
    few = eng.run(ids[-43:], traj=True, final=True)
    np.testing.assert_array_equal(few.beta_final, res.beta_final[-43:])
    np.testing.assert_array_equal(few.traj_m2, res.traj_m2[-43:])
    for k, v in (("sum_n", np.abs(few.traj) ** 2), ("sum_beta", few.traj)):
        assert rel_err(getattr(few, k), v.sum(axis=0)) < 1e-12
    eng.close()
