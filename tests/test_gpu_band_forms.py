"""The banded kernel's forms -- site parameters that differ only in the energies
or in everything, batches below and above two waves per SIMD -- at two to eight
sites per lane and half-widths one to three, open and cyclic: against the FP64
oracle, and the same trajectory from either batch size bit for bit."""
import numpy as np
import pytest

import oracle
from helpers import FP32_BAR, rel_err
from pincosimulator_amd import Engine, System
from test_gpu_band import band_matrix, matrix_spec
from test_gpu_mfma import lieb_disordered

pytestmark = pytest.mark.gpu

COUPLINGS = [band_matrix(n, w, cyc, 31 * n + w) for n, w, cyc in
             ((100, 1, False), (128, 2, True), (90, 2, False), (256, 3, True), (200, 1, False), (330, 3, False),
              (384, 2, True), (512, 2, True), (500, 3, False))] + [lieb_disordered(128, pbc=True)]


@pytest.mark.parametrize("C", COUPLINGS, ids=[f"{k}-{c.shape[0]}" for k, c in enumerate(COUPLINGS)])
@pytest.mark.parametrize("uniform", [True, False])
def test_forms_match_oracle(C, uniform):
    n = C.shape[0]
    spec = matrix_spec(C, t_end=0.05, frame_steps=5)
    if not uniform:
        spec["F"] = 1.2 * np.exp(1j * np.linspace(0, 3, n))
        spec["U"] = np.linspace(0.05, 0.1, n) + 0.02j
    ids = np.arange(2500, dtype=np.uint64) * 3
    print(f"band {n} sites, uniform {uniform}", flush=True)
    eng = Engine(System(**spec), precision=32, kernel="band")
    out = eng.run(ids, final=True).beta_final
    p = dict(spec, lattice=oracle.LAT_DENSE, E=spec["omega"])
    for j in (0, 1024, 2499):
        assert rel_err(out[j], oracle.run_trajectory(p, int(ids[j]))[1]) < FP32_BAR
    np.testing.assert_array_equal(eng.run(ids[2400:], final=True).beta_final, out[2400:])
    eng.close()
