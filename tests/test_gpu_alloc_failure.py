"""Allocations that fail (tests/native/alloc_fail.c returns the error in the library's
process; the GPU does not see them): calls that have another way take it with the same
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
from pincosimulator_amd import Engine, System
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
