"""The step kernel of small lattices in small batches (the noise formed ahead of the
steps): one to four sites per lane and the edges between them, a single site pair,
odd and even rows, chains, uniform, varying and drawn parameters, step counts below,
at and above a chunk of noise and its remainders, FP32 and FP64; against the FP64
oracle, and the same trajectories from a batch on the other side of the batch-size
rule (two to 16 trajectories per CU) bit for bit."""
import numpy as np
import pytest
import torch

import oracle
from helpers import FP32_BAR, c2_spec, oracle_params, rel_err, system
from pincosimulator_amd import Engine
from test_gpu_nn_forms import site_forms

pytestmark = pytest.mark.gpu

SHAPES = [(1, 2), (3, 3), (4, 4), (1, 63), (8, 8), (5, 13), (1, 127), (2, 64), (3, 43), (10, 25), (1, 255), (16, 16)]


@pytest.mark.parametrize("nx,ny", SHAPES, ids=[f"{a}x{b}" for a, b in SHAPES])
@pytest.mark.parametrize("precision", [32, 64])
def test_small_lattices_match_oracle(nx, ny, precision):
    n = nx * ny
    cus = torch.cuda.get_device_properties(0).multi_processor_count
    many = cus * (2 if n > 128 else 16 if precision == 32 else 4 if n > 64 else 8) + 1
    for k, (name, form) in enumerate(site_forms(n).items()):
        frame_steps = (131, 64, 1, 8, 100, 17)[k]
        spec = c2_spec(**dict(dict(nx=nx, ny=ny, U=0.08 + 0.02j, F=0.8 + 0.3j, omega=0.3, J=0.7, dt=0.005,
                                   t_end=0.005 * (131 + 0.25), seed=n + k, frame_steps=frame_steps), **form))
        ids = np.arange(many, dtype=np.uint64) * 5 + 2
        print(f"{nx}x{ny}, FP{precision}, {name}", flush=True)
        eng = Engine(system(spec), precision=precision, kernel="generic")
        few = eng.run(ids[-20:], final=True).beta_final
        for j in (0, 19):
            err = rel_err(few[j], oracle.run_trajectory(oracle_params(spec), int(ids[many - 20 + j]))[1])
            assert err < (FP32_BAR if precision == 32 else 1e-9)
        np.testing.assert_array_equal(eng.run(ids, final=True).beta_final[-20:], few)
        eng.close()
