"""Small systems in small batches store several frames per launch: the same run taken
segment by segment (one frame per launch), in uneven pieces and at once -- with and
without the states, with steps after the last frame, more frames than a launch takes
(64), single-step frames, matrix hopping -- gives the same states and means bit for
bit and the same sums to rounding (the slots of a sum differ)."""
import numpy as np
import pytest

from helpers import c2_spec, rel_err, system
from pincosimulator_amd import Engine, System
from test_gpu_sparse import sparse_matrix, spec_of

pytestmark = pytest.mark.gpu

RUNS = {"chain": (dict(nx=1, ny=64, dt=0.01, frame_steps=7, t_end=0.01 * 36.25), {}),
        "single steps": (dict(nx=5, ny=13, dt=0.01, frame_steps=1, t_end=0.01 * 140.25), {}),
        "no first frame": (dict(nx=4, ny=4, dt=0.01, frame_steps=70, t_end=0.01 * 285.25), dict(store_initial=False)),
        "drawn": (dict(nx=12, ny=14, dt=0.01, frame_steps=3, t_end=0.01 * 30.25,
                       F={"base": 1.0, "noise": ("gaussian", 0.3)}), {}),
        "matrix": (72, {})}


@pytest.mark.parametrize("name", list(RUNS))
@pytest.mark.parametrize("precision", [32, 64])
@pytest.mark.parametrize("traj", [False, True])
def test_frames_in_groups(name, precision, traj):
    kw, opt = RUNS[name]
    spec = spec_of(sparse_matrix(kw, 3, 5), frame_steps=9, t_end=0.005 * 50.25) if name == "matrix" else c2_spec(**kw)
    print(f"{name}, FP{precision}, states {traj}", flush=True)
    eng = Engine(System(**spec) if name == "matrix" else system(spec), precision=precision, kernel="generic")
    res = []
    for piece in (1, 3, 10 ** 6):
        info = eng.begin(np.arange(37, dtype=np.uint64) * 9, traj=traj, final=True, **opt)
        while info["segments_done"] < info["n_segments"]:
            eng.advance(piece)
            eng.sync()
            info = eng.info()
        res.append(eng.read())
    eng.close()
    assert res[0].n_frames > 1
    for r in res[1:]:
        for k in ("beta_final", "traj_m2", "traj_m4") + (("traj",) if traj else ()):
            np.testing.assert_array_equal(getattr(r, k), getattr(res[0], k))
        for k in ("sum_n", "sum_n2", "sum_nk", "sum_beta"):
            assert rel_err(getattr(r, k), getattr(res[0], k)) < 1e-13 or not np.any(getattr(res[0], k))
