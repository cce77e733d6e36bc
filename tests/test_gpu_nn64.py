"""The FP64 step kernel of site-uniform lattices with even rows, 257 to 4096 sites: at
the edges of its workgroup shapes (partly filled waves, one or two pairs per thread,
rows without x neighbours), odd and even step counts, a real and a complex U, batches
below and above its grid, against the FP64 oracle; the same trajectory from a batch on
the other side of the batch-size rule bit for bit."""
import numpy as np
import pytest

import oracle
from helpers import c2_spec, oracle_params, rel_err, system
from pincosimulator_amd import Engine

pytestmark = pytest.mark.gpu

SHAPES = [(1, 258), (2, 130), (16, 32), (1, 514), (27, 38), (32, 32), (2, 514), (3, 342), (64, 32), (1, 2050),
          (36, 58), (50, 80), (64, 64)]


@pytest.mark.parametrize("nx,ny", SHAPES, ids=[f"{a}x{b}" for a, b in SHAPES])
@pytest.mark.parametrize("U", [0.1, 0.08 + 0.02j])
def test_nn64_matches_oracle(nx, ny, U):
    spec = c2_spec(nx=nx, ny=ny, U=U, F=0.8 + 0.3j, J=0.7, dt=0.01, t_end=0.06, seed=nx + ny, frame_steps=3)
    ids = np.arange(2050, dtype=np.uint64) * 5 + 1
    print(f"nn64 {nx}x{ny}, U {U}", flush=True)
    eng = Engine(system(spec), precision=64, kernel="generic")
    out = eng.run(ids, final=True).beta_final
    for j in (0, 2049):
        assert rel_err(out[j], oracle.run_trajectory(oracle_params(spec), int(ids[j]))[1]) < 1e-9
    few = eng.run(ids[-30:], final=True).beta_final  # above 2048 sites: the LDS kernel's own launch
    np.testing.assert_array_equal(few, out[-30:])
    eng.close()
