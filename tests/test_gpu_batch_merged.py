"""The batch form with one launch per phase over every instance (the default up to 4,194,304
particles): each instance bit-equal to the same instance stepped alone, at batch totals on both
sides of the sizes at which the sweeps' split changes, with instances that cannot take bond records
in the same batch, and after the autotuner has chosen."""
import sys

import numpy as np
import pytest

from morphogenesis_amd import _ffi as F
from morphogenesis_amd import scenes
from tests.helpers import assert_bits_equal

pytestmark = pytest.mark.gpu

STATE = [F.FPOS, F.FVEL, F.FVEVAL, F.FPRESS, F.FDENSITY, F.FGCELL, F.FGNDX, F.FELASTIDX, F.FCONC, F.FEPIGEN,
         F.FPARTICLE_ID, F.FBIN_COUNT, F.FBIN_OFFSET]


def open_scene(sc):
    from morphogenesis_amd.fluid_system import FluidSystem

    sim = FluidSystem(sc.n, sc.b)
    sim.load_scene(sc)
    sim.Run2PhysicalSort()
    return sim


@pytest.mark.parametrize("dims,b,steps", [
    ([(1, 1, 1), (4, 4, 4), (5, 13, 1), (9, 9, 9)], [4, 6, 32, 32], 5),      # every sweep by rows
    ([(32, 32, 32), (20, 21, 40), (3, 5, 7)], [12, 6, 4], 4),                # 49,673: pressure in threes
    ([(32, 32, 40), (30, 30, 20), (8, 8, 8)], [6, 12, 32], 3),               # 59,472: a lane per diffusing particle
    ([(48, 48, 60), (20, 20, 24)], [6, 6], 2),                               # 147,840: a lane in the force too
    ([(9, 9, 9), (10, 9, 8)], [0, 8], 4),                                    # no bond slots beside bonds
])
def test_merged_form_matches_single(built, dims, b, steps):
    from morphogenesis_amd.batch import Batch

    scs = [scenes.tissue(b=bb, seed=40 + k, dims=d) for k, (d, bb) in enumerate(zip(dims, b))]
    for sc in scs:
        sc.buffers[F.FVEL][:, :3] = np.random.default_rng(sc.n).normal(0, 3.0, (sc.n, 3))
    print("case: merged batch", [sc.n for sc in scs], "B", b, flush=True)
    sys.stdout.flush()
    together, alone = [open_scene(sc) for sc in scs], [open_scene(sc) for sc in scs]
    bat = Batch(together)
    flags = F.STEP_GENES
    bat.step(steps, scs[0].dt, flags | F.STEP_GRAPH)
    bat.step(1, scs[0].dt, flags)
    bat.sync()
    assert bat.launch_config() == (0, 0)
    for k, sim in enumerate(alone):
        sim.step(steps + 1, scs[0].dt, flags)
        for buf in STATE:
            assert_bits_equal(together[k].download(buf), sim.download(buf), f"instance {k}: {F.BUFFER_NAMES[buf]}")
    # switching the form between graph replays keeps every instance on its course
    for form in (True, False):
        bat.set_persistent(form)
        bat.step(2, scs[0].dt, flags | F.STEP_GRAPH)
    bat.sync()
    for k, sim in enumerate(alone):
        sim.step(4, scs[0].dt, flags)
        assert_bits_equal(together[k].download(F.FPOS), sim.download(F.FPOS), f"instance {k}: FPOS after switches")
    bat.autotune(1, scs[0].dt, flags)
    bat.step(2, scs[0].dt, flags | F.STEP_GRAPH)
    bat.sync()
    bat.close()
