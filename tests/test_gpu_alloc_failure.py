"""Allocations that fail (tests/native/alloc_fail.c asks the runtime for too much in the library's
process, which the host refuses): calls that have another way take it with the same
results, the others return an error and leave a context that later calls can use."""
import os
import subprocess
import sys
import textwrap

import pytest

from conftest import ROOT

pytestmark = pytest.mark.gpu

HEAD = """
import ctypes, sys
sys.path[:0] = [{root!r}, {tests!r}]
fail = ctypes.CDLL({so!r}, mode=ctypes.RTLD_GLOBAL)
fail.fail_device_above.argtypes = [ctypes.c_size_t]
import numpy as np
from pincosimulator_amd import Engine, Sweep
from pincosimulator_amd._lib import TWMCError
from pincosimulator_amd.mlp import MLP
from helpers import c2_spec, system
"""


@pytest.fixture(scope="module")
def run(tmp_path_factory):
    so = str(tmp_path_factory.mktemp("alloc") / "liballoc_fail.so")
    subprocess.check_call(["gcc", "-O1", "-shared", "-fPIC", "-o", so, os.path.join(ROOT, "tests/native/alloc_fail.c"),
                           "-ldl"])

    def child(body):
        code = HEAD.format(root=ROOT, tests=os.path.join(ROOT, "tests"), so=so) + textwrap.dedent(body)
        r = subprocess.run([sys.executable, "-u", "-c", code], capture_output=True, text=True, timeout=100)
        assert r.returncode == 0 and r.stdout.rstrip().endswith("done"), r.stdout + r.stderr

    return child


def test_read_back_without_pinned_memory(run):
    """64 trajectories of 64x64, three stored frames: 6.3 MB."""
    run("""
    spec = c2_spec(frame_steps=3, t_end=0.002 * 6.25)
    ids = np.arange(64, dtype=np.uint64)
    out = []
    for on in (1, 0):
        fail.fail_pinned(on)
        eng = Engine(system(spec), precision=32)
        out.append(eng.run(ids, traj=True, final=True))
        eng.close()
        assert fail.failures() > 0
    np.testing.assert_array_equal(out[0].traj, out[1].traj)
    np.testing.assert_array_equal(out[0].beta_final, out[1].beta_final)
    assert np.all(np.any(out[0].traj != 0, axis=2))
    print("done")
    """)


def test_training_without_pinned_memory(run):
    run("""
    rng = np.random.default_rng(2)
    x, t = (rng.normal(size=(300, k)).astype(np.float32) for k in (5, 7))
    out = []
    for on in (1, 0):
        fail.fail_pinned(on)
        m = MLP(5, 7, n_hidden=20, n_hidden_layers=2, seed=4)
        m.train(x[:50], t[:50], epochs=3, batch=16)
        m.train(x, t, epochs=3, batch=16)  # longer orders
        out.append(m.params)
        fail.fail_pinned(0)
        m.close()
        assert fail.failures() > 0
    np.testing.assert_array_equal(*out)
    print("done")
    """)


def test_error_is_reported_once(run):
    run("""
    def fails(call):
        fail.fail_device_above(100000)
        try:
            call()
            raise SystemExit("no error")
        except TWMCError as e:
            assert "memory" in str(e)
        fail.fail_device_above(1 << 40)

    m = MLP(5, 7, n_hidden=20, n_hidden_layers=2, seed=4)
    x = np.ones((4000, 5), dtype=np.float32)
    fails(lambda: m.forward(x))
    assert np.all(np.isfinite(m.forward(x[:9])))
    m.close()
    spec = c2_spec(nx=4, ny=8, frame_steps=5, t_end=0.002 * 15.25)
    eng = Engine(system(spec), precision=32)
    fails(lambda: eng.begin(np.arange(5000)))
    assert np.all(np.isfinite(eng.run(np.arange(3)).sum_n))
    eng.close()
    point = dict(nx=1, ny=64, gamma=1.0, J=1.0, U=0.1, F=1.0, traj_id0=0)
    fails(lambda: Sweep([dict(point, n_traj=1000)], 0.005, 10, 3))
    sw = Sweep([dict(point, n_traj=10)], 0.005, 10, 3)
    assert np.all(np.isfinite(sw.run(0.2, graph=False)["m2"][0]))
    sw.close()
    print("done")
    """)


@pytest.mark.parametrize("hidden", [20, 300])
def test_network_after_a_failed_call(run, hidden):
    """A gradient over 20000 rows fails at its larger buffers; the smaller batches after it."""
    run(f"""
    rng = np.random.default_rng(2)
    x, t = (rng.normal(size=(20000, k)).astype(np.float32) for k in (5, 7))
    m = MLP(5, 7, n_hidden={hidden}, n_hidden_layers=2, seed=4)
    first = m.loss_grad(x[:64], t[:64])
    fail.fail_device_above(1000000)
    for call in (lambda: m.loss_grad(x, t), lambda: m.forward(x), lambda: m.loss_grad(x, t)):
        try:
            call()
            raise SystemExit("no error")
        except TWMCError:
            pass
    assert fail.failures() == 3
    again = m.loss_grad(x[:64], t[:64])
    np.testing.assert_array_equal(first[1], again[1])
    assert first[0] == again[0]
    np.testing.assert_allclose(m.forward(x[:64]), m.forward(x[:70])[:64], rtol=0, atol=0)
    fail.fail_device_above(1 << 40)
    assert np.all(np.isfinite(m.loss_grad(x, t)[1]))
    m.close()
    print("done")
    """)


def test_sweep_after_a_failed_call(run):
    """A stacking that is refused or fails, and a run whose outputs do not fit, leave the sweep as it was."""
    run("""
    point = dict(nx=1, ny=64, gamma=1.0, J=1.0, U=0.1, F=1.0, traj_id0=0, n_traj=1000)
    sw = Sweep([point, dict(point, nx=4, ny=8)], 0.005, 10, 3)
    tb = sw.batching()
    first = sw.run(0.2, graph=False)
    for limit, call in ((4000, lambda: sw.set_batching([1, 1])), (1 << 40, lambda: sw.set_batching([2, 1000])),
                        (100000, lambda: sw.run(2.0, graph=False))):
        fail.fail_device_above(limit)
        try:
            call()
            raise SystemExit("no error")
        except TWMCError:
            pass
        fail.fail_device_above(1 << 40)
        assert sw.batching() == tb
        again = sw.run(0.2, graph=False)
        for a, b in zip(first["m2"] + first["m4"], again["m2"] + again["m4"]):
            np.testing.assert_array_equal(a, b)
        # added atomically, 64000 terms in any order
        np.testing.assert_allclose(first["ksum"], again["ksum"], rtol=1e-11)
    sw.close()
    print("done")
    """)


def test_no_batch_after_a_failed_begin(run):
    run("""
    spec = c2_spec(nx=4, ny=8, frame_steps=5, t_end=0.002 * 15.25)
    eng = Engine(system(spec), precision=32)
    want = eng.run(np.arange(3), final=True).beta_final
    for good in (3, 40):
        eng.begin(np.arange(good))
        fail.fail_device_above(100000)
        for call in (lambda: eng.begin(np.arange(5000)), lambda: eng.advance(1), eng.read):
            try:
                call()
                raise SystemExit("no error")
            except TWMCError as e:
                assert "memory" in str(e) or "no active batch" in str(e)
        np.testing.assert_array_equal(eng.run(np.arange(3), final=True).beta_final, want)
        fail.fail_device_above(1 << 40)
    eng.close()
    print("done")
    """)


def test_frames_one_by_one_without_memory_for_groups(run):
    """256 trajectories of 64 sites, 20 frames: 0.7 MB of partial sums and 0.3 MB of states a frame."""
    run("""
    spec = c2_spec(nx=1, ny=64, frame_steps=4, t_end=0.002 * 76.25)
    out = []
    for bytes in (1000000, 1 << 40):
        fail.fail_device_above(bytes)
        eng = Engine(system(spec), precision=64, kernel="generic")
        out.append(eng.run(np.arange(256), final=True))
        eng.close()
    assert out[0].n_frames == 20 and fail.failures() == 1
    for k in ("beta_final", "traj_m2", "sum_n", "sum_nk"):
        np.testing.assert_array_equal(getattr(out[0], k), getattr(out[1], k))
    print("done")
    """)
