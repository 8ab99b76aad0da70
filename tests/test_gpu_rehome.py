"""Re-homing on the device: the permutation, the numbers given to particles outside the sorted
region, and the bond rows, at the edges of its 4,096-word tiles, with particles parked and dropped
outside the window, again after a later sort. Every buffer bit-equal to the oracle."""
import sys

import numpy as np
import pytest

from morphogenesis_amd import _ffi as F
from morphogenesis_amd import scenes
from tests.test_gpu_parity import compare_all, pair

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("dims,reserve,dropped,b", [
    ((1, 1, 1), 2, 0, 2),
    ((15, 16, 17), 15, 9, 6),    # 4,095
    ((16, 16, 16), 0, 0, 1),     # 4,096, all inside
    ((16, 16, 16), 1, 0, 4),     # 4,097
    ((16, 16, 32), 1, 200, 8),   # 8,193
    ((12, 11, 10), 0, 1320, 4),  # nobody inside
])
def test_rehoming(built, dims, reserve, dropped, b):
    sc = scenes.tissue(b=b, seed=9, dims=dims, reserve=reserve)
    print("case: re-homing", sc.n, "reserve", reserve, "dropped", dropped, "B", b, flush=True)
    sys.stdout.flush()
    rng = np.random.default_rng(1)
    live = dims[0] * dims[1] * dims[2]
    sc.buffers[F.FVEL][:, :3] = rng.normal(0, 2.0, (sc.n, 3))
    sc.buffers[F.FPOS][rng.choice(live, dropped, replace=False), 0] = 0.4  # outside the window
    g, o = pair(sc)
    for sim in (g, o):
        sim.Run2PhysicalSort()
        sim.step(3, sc.dt, sc.flags)
    compare_all(g, o, "steps after the first sort")
    for sim in (g, o):
        sim.Run2InnerPhysicalLoop(sc.dt)
        sim.Run2PhysicalSort()
        sim.step(4, sc.dt, sc.flags | (F.STEP_GRAPH if sim is g else 0))
    compare_all(g, o, "steps after another sort")
