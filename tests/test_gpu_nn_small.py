"""The nearest-neighbour step kernel at 65 to 128 sites (one wave per trajectory), whose
batches are above the small-batch kernel's: odd rows and, FP32, varying parameters, a
partly filled last pair and wave; against the FP64 oracle."""
import numpy as np
import pytest

import oracle
from helpers import FP32_BAR, c2_spec, oracle_params, rel_err, system
from pincosimulator_amd import Engine
from test_gpu_nn_forms import site_forms

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("nx,ny", [(5, 13), (1, 65), (2, 33), (1, 127), (8, 16), (3, 41)])
@pytest.mark.parametrize("precision", [32, 64])
def test_one_wave_lattices_match_oracle(nx, ny, precision):
    for k, (name, form) in enumerate(site_forms(nx * ny).items()):
        spec = c2_spec(**dict(dict(nx=nx, ny=ny, U=0.08 + 0.02j, F=0.8 + 0.3j, omega=0.3, J=0.7, dt=0.005,
                                   t_end=0.005 * (8.25 + k % 2), seed=nx * ny + k, frame_steps=3), **form))
        ids = np.arange(9001, dtype=np.uint64) * 7 + 3
        print(f"{nx}x{ny}, FP{precision}, {name}", flush=True)
        eng = Engine(system(spec), precision=precision, kernel="generic")
        out = eng.run(ids, final=True).beta_final
        eng.close()
        for j in (0, 4500, 9000):
            err = rel_err(out[j], oracle.run_trajectory(oracle_params(spec), int(ids[j]))[1])
            assert err < (FP32_BAR if precision == 32 else 1e-9)
