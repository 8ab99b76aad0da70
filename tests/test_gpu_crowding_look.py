"""Models above 57,344 particles choose how to step crowded cells (a list of dense groups; the pressure
with a lane per particle) by a look at their cells, when the homes are numbered and every 256 steps:
the choice follows particles that crowd, or part, in between; and the steps before and after it give
the same bits as those of a model whose homes are numbered anew."""
import ctypes as C
import sys

import numpy as np
import pytest

from morphogenesis_amd import _ffi as F
from morphogenesis_amd.fluid_system import FluidSystem
from tests.helpers import assert_bits_equal
from tests.test_gpu_dense import with_drop

pytestmark = pytest.mark.gpu

DT = 1e-6


def say(*a):
    print(*a, flush=True)
    sys.stdout.flush()


def crowding(sim):
    row, crowded, listed = C.c_uint32(), C.c_int(), C.c_uint32()
    assert sim.lib.mg_debug_crowding(sim.h, C.byref(row), C.byref(crowded), C.byref(listed)) == F.MG_OK
    return row.value, crowded.value, listed.value


def scale(sim, f, only=slice(None)):
    """The particles' distances from the middle scaled by f, without a sort by the program (which would
    number the homes): the next step bins them."""
    p = sim.download(F.FPOS)
    mid = p[only, :3].mean(0)
    p[only, :3] = mid + (p[only, :3] - mid) * np.float32(f)
    sim.upload(F.FPOS, p)
    sim.step(1, DT, F.STEP_GENES)


@pytest.mark.parametrize("drop", [0, 1000])
def test_choice_follows_the_particles(built, drop):
    sc = with_drop((56, 56, 56), 4, True, 0.5, drop)
    sc.buffers[F.FVEL][:] = 0
    sc.buffers[F.FVEVAL][:] = 0
    sc.params.diff_scale = 1e-5  # hundreds of neighbours: concentrations stay finite
    say("case: crowding looked at,", sc.n, "with a drop of", drop)
    sim, ref = FluidSystem(sc.n, sc.b), FluidSystem(sc.n, sc.b)
    flags = F.STEP_GENES | F.STEP_GRAPH
    for s in (sim, ref):
        s.load_scene(sc)
        s.Run2PhysicalSort()
        s.step(2, DT, flags)
    row, crowded, listed = crowding(sim)
    assert crowded == 0 and (row >= 64 and listed > 0 if drop else (row, listed) == (0, 0))
    for f, want in ((0.55, 1), (1 / 0.55, 0)):
        for s in (sim, ref):
            scale(s, f)
        ref.Run2PhysicalSort()  # numbers the homes at its next step
        for _ in range(7):
            for s in (sim, ref):
                s.step(50, DT, flags)
        got = crowding(sim)
        say("scaled by", f, "row, crowded, listed:", got, "homes renumbered:", crowding(ref))
        assert got[1] == want and got == crowding(ref)
        if want:
            assert got[2] == 0  # crowded throughout: nothing is listed
        for buf in (F.FPOS, F.FVEL, F.FPRESS, F.FCONC, F.FEPIGEN, F.FGCELL):
            assert_bits_equal(sim.download(buf), ref.download(buf), f"scaled by {f}: {F.BUFFER_NAMES[buf]}")
    for s in (sim, ref):
        s.close()


@pytest.mark.parametrize("n_side,want", [(56, 1), (54, 0)])  # 175,616 and 157,464: the rule's line between
def test_phase_calls_choose_too(built, n_side, want):
    """A program of phase calls alone numbers no homes; its pressure passes look by themselves."""
    sc = with_drop((n_side,) * 3, 0, False, 0.28, 0)
    say("case: phase calls look,", sc.n)
    sim = FluidSystem(sc.n, sc.b)
    sim.load_scene(sc)
    sim.Run2PhysicalSort()
    assert crowding(sim)[1] == 0
    sim.Run2InnerPhysicalLoop(DT)
    assert crowding(sim)[1] == want
    sim.Run2PhysicalSort()
    p = sim.download(F.FPOS)
    mid = p[:, :3].mean(0)
    p[:, :3] = mid + (p[:, :3] - mid) * np.float32(0.5 / 0.28)
    sim.upload(F.FPOS, p)
    for _ in range(257):
        sim.Run2PhysicalSort()
        sim.ComputePressureCL()
    assert crowding(sim)[1] == 0
    sim.close()
