"""The nearest-neighbour step kernel's other forms, 129 to 4096 sites: rows of odd
length (pairs across two rows, a last site without a partner), chains, and energies
or drives that vary from site to site or are drawn per trajectory, complex or not, in
FP32 and FP64, at the edges of the workgroup shapes; against the FP64 oracle, and the
same trajectory from a small batch bit for bit."""
import numpy as np
import pytest

import oracle
from helpers import FP32_BAR, c2_spec, oracle_params, rel_err, system
from pincosimulator_amd import Engine

pytestmark = pytest.mark.gpu

SHAPES = [(1, 129), (1, 130), (5, 51), (2, 128), (3, 171), (2, 255), (1, 513), (31, 33), (32, 32), (23, 89), (2, 1024),
          (1, 2049), (50, 81), (45, 91), (64, 64)]


def site_forms(n):
    rng = np.random.default_rng(n)
    return {"uniform": {},
            "omega": dict(omega=0.4 * rng.standard_normal(n) + 0.05j * rng.standard_normal(n)),
            "omega drawn": dict(omega={"base": 0.3, "noise": ("gaussian", 0.2 + 0.05j)}),
            "F": dict(F=1.2 * np.exp(1j * rng.uniform(0, 6, n))),
            "F drawn": dict(F={"base": 0.9 - 0.4j, "noise": ("uniform", 0.3)}),
            "F and U": dict(F=1.2 * np.exp(1j * rng.uniform(0, 6, n)), U=np.linspace(0.05, 0.1, n) + 0.02j)}


@pytest.mark.parametrize("nx,ny", SHAPES, ids=[f"{a}x{b}" for a, b in SHAPES])
@pytest.mark.parametrize("precision", [32, 64])
def test_forms_match_oracle(nx, ny, precision):
    for k, (name, form) in enumerate(site_forms(nx * ny).items()):
        spec = c2_spec(**dict(dict(nx=nx, ny=ny, U=0.08 + 0.02j, F=0.8 + 0.3j, omega=0.3, J=0.7, dt=0.005,
                                   t_end=0.005 * (8.25 + k % 2), seed=nx * ny + k, frame_steps=3), **form))
        ids = np.arange(1100 if nx * ny > 1000 else 2300, dtype=np.uint64) * 7 + 3
        print(f"{nx}x{ny}, FP{precision}, {name}", flush=True)
        eng = Engine(system(spec), precision=precision)
        out = eng.run(ids, final=True).beta_final
        for j in (0, len(ids) // 2, len(ids) - 1):
            err = rel_err(out[j], oracle.run_trajectory(oracle_params(spec), int(ids[j]))[1])
            assert err < (FP32_BAR if precision == 32 else 1e-9)
        np.testing.assert_array_equal(eng.run(ids[-20:], final=True).beta_final, out[-20:])
        eng.close()
