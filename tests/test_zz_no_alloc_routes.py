"""Allocation-free stepping on the launches that test_zz_no_alloc.py's small batches do not
reach, checked the same way: work queues with more trajectories than workgroups (64x64,
and the nearest-neighbour kernel with odd rows, one varying parameter, FP64), matrix
hopping in a wave's registers and with the noise ahead, 32 trajectories per matrix-core
workgroup; each time a smaller second call, whose queue and tables overwrite the first's."""
import numpy as np
import pytest

import test_zz_no_alloc as base
from test_gpu_mfma import c3_spec

pytestmark = pytest.mark.gpu


def lieb(cells):
    return dict(c3_spec(cells=cells, t_end=1.0, frame_steps=30))


CASES = [("stencil64", 32, base.square(64, 64, 30), 1100, 600),
         ("generic", 64, base.square(64, 64, 30), 600, 513),
         ("generic", 32, base.square(27, 41, 30), 3000, 1500),
         ("generic", 64, dict(base.square(16, 18, 30), F=1.4 * np.exp(0.01j * np.arange(288))), 4500, 300),
         ("generic", 64, lieb(24), 2100, 70),
         ("generic", 64, lieb(128), 1000, 600),
         ("mfma", 32, lieb(128), 4200, 33)]


@pytest.mark.parametrize("kernel,prec,spec,b1,b2", CASES,
                         ids=[f"{c[0]}-fp{c[1]}-{c[2]['nx']}x{c[2]['ny']}-{c[3]}" for c in CASES])
def test_noalloc_by_route(kernel, prec, spec, b1, b2):
    base.test_noalloc_equals_the_allocating_entry_point(kernel, prec, spec, b1, b2)
