"""The 64x64 step kernel where its launch can go wrong: one, two and three steps
per launch (two per loop pass, and a remainder), real and complex interaction,
more trajectories than workgroups (512 on 256 CUs: a second trajectory after the
first), against the FP64 oracle; and the same trajectory from batches of
different sizes bit for bit."""
import numpy as np
import pytest

import oracle
from helpers import FP32_BAR, c2_spec, rel_err, system
from pincosimulator_amd import Engine

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("U", [0.05, 0.05 + 0.02j])
@pytest.mark.parametrize("frame_steps", [1, 2, 3])
def test_steps_per_launch(frame_steps, U):
    spec = c2_spec(U=U, frame_steps=frame_steps, t_end=0.002 * 6, seed=5)
    print(f"stencil64 {frame_steps} steps per launch, U = {U}", flush=True)
    eng = Engine(system(spec), precision=32)
    ids = np.arange(3) + 7
    res = eng.run(ids, traj=True)
    eng.close()
    assert res.kernel == "stencil64" and res.n_steps == 6
    p = dict(spec, lattice=oracle.LAT_FFT)
    for j, t in enumerate(ids):
        assert rel_err(res.traj[j], oracle.run_trajectory(p, int(t))[0]) < FP32_BAR


def test_batches_of_any_size_give_the_same_bits():
    spec = c2_spec(frame_steps=5, t_end=0.02, seed=6)
    ids = np.arange(1300, dtype=np.uint64)
    print("stencil64 1300 trajectories", flush=True)
    eng = Engine(system(spec), precision=32)
    whole = eng.run(ids, final=True).beta_final
    p = dict(spec, lattice=oracle.LAT_FFT)
    for t in (0, 511, 512, 1023, 1024, 1299):
        assert rel_err(whole[t], oracle.run_trajectory(p, t)[1]) < FP32_BAR
    np.testing.assert_array_equal(eng.run(ids[500:540], final=True).beta_final, whole[500:540])
    np.testing.assert_array_equal(eng.run(ids[:1], final=True).beta_final, whole[:1])
    eng.close()
