"""FP64 lattices with even rows whose step launch follows the batch: up to 256 sites with
a varying parameter (from 12 trajectories per CU the nearest-neighbour kernel), 257 to
512 uniform ones (from four); either side of the line against the FP64 oracle, and the
same trajectories bit for bit."""
import numpy as np
import pytest
import torch

import oracle
from helpers import c2_spec, oracle_params, rel_err, system
from pincosimulator_amd import Engine
from test_gpu_nn_forms import site_forms

pytestmark = pytest.mark.gpu

CASES = [(nx, ny, f) for nx, ny in ((1, 130), (16, 16)) for f in ("omega", "omega drawn", "F drawn")] + \
    [(1, 258, "uniform"), (16, 24, "uniform"), (1, 512, "uniform")]


@pytest.mark.parametrize("nx,ny,form", CASES, ids=[f"{a}x{b} {f}" for a, b, f in CASES])
def test_batches_agree(nx, ny, form):
    n = nx * ny
    spec = c2_spec(**dict(dict(nx=nx, ny=ny, U=0.08 + 0.02j, F=0.8 + 0.3j, omega=0.3, J=0.7, dt=0.005,
                               t_end=0.005 * 9.25, seed=n, frame_steps=3), **site_forms(n)[form]))
    cus = torch.cuda.get_device_properties(0).multi_processor_count
    line = cus * (12 if n <= 256 else 4)
    ids = np.arange(line, dtype=np.uint64) * 7 + 3
    print(f"{nx}x{ny}, {form}", flush=True)
    eng = Engine(system(spec), precision=64)
    many = eng.run(ids, final=True).beta_final
    for j in (0, line - 1):
        assert rel_err(many[j], oracle.run_trajectory(oracle_params(spec), int(ids[j]))[1]) < 1e-9
    np.testing.assert_array_equal(eng.run(ids[1:], final=True).beta_final, many[1:])
    eng.close()
