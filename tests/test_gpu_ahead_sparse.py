"""Matrix hopping with few nonzeros per column in small batches (the noise formed ahead
of the steps): one to eight sites per lane and the edges between them, one to six
nonzeros, a single site, drawn and fixed parameters, step counts around the noise's
chunks, FP32 and FP64; against the FP64 oracle, and the same trajectories from a batch
on the sparse kernel's side of the batch-size rule bit for bit."""
import numpy as np
import pytest
import torch

import oracle
from helpers import FP32_BAR, rel_err
from pincosimulator_amd import Engine, System
from test_gpu_sparse import sparse_matrix, spec_of

pytestmark = pytest.mark.gpu

CASES = [(1, 1), (2, 1), (3, 3), (63, 3), (64, 6), (65, 4), (127, 6), (128, 3), (129, 6), (200, 2), (255, 3), (256, 5),
         (257, 3), (384, 2), (509, 3), (512, 3)]


@pytest.mark.parametrize("n,most", CASES, ids=[f"{n}-{m}" for n, m in CASES])
@pytest.mark.parametrize("precision", [32, 64])
def test_small_batches_match_oracle(n, most, precision):
    cus = torch.cuda.get_device_properties(0).multi_processor_count
    many = cus * (8 if n <= 128 else 2 if n <= 256 or precision == 64 else 1) + 1
    for k, drawn in enumerate((True, False)):
        spec = spec_of(sparse_matrix(n, most, 7 * n + most), frame_steps=(130, 41)[k], t_end=0.005 * 130.25)
        if drawn:
            spec["omega"] = {"base": spec["omega"], "noise": ("gaussian", 0.2)}
        ids = np.arange(many, dtype=np.uint64) * 3 + 4
        print(f"{n} sites, {most} nonzeros, FP{precision}, drawn {drawn}", flush=True)
        eng = Engine(System(**spec), precision=precision, kernel="generic")
        few = eng.run(ids[-20:], final=True).beta_final
        p = dict(spec, lattice=oracle.LAT_DENSE, E=spec["omega"])
        for j in (0, 19):
            err = rel_err(few[j], oracle.run_trajectory(p, int(ids[many - 20 + j]))[1])
            assert err < (FP32_BAR if precision == 32 else 1e-9)
        if precision == 64 or drawn:  # FP32 with fixed parameters: the LDS kernel for any batch
            np.testing.assert_array_equal(eng.run(ids, final=True).beta_final[-20:], few)
        eng.close()
