"""Diffusion split by rows of groups with crowded rows (`diffuse_crowded`): bit-equal to the oracle where
the masks take one round of LDS and several, where crowded groups and others share a model, at rows
about the size from which a group counts as crowded, for one, two and four float4 groups of
concentrations, in the fused step and the phase calls; and its time beside the pressure pass, which
tests the same candidates."""
import ctypes as C
import sys

import numpy as np
import pytest

from morphogenesis_amd import _ffi as F
from morphogenesis_amd import scenes
from morphogenesis_amd.fluid_system import FluidSystem
from tests.test_gpu_dense import with_drop
from tests.test_gpu_parity import compare_all, pair

pytestmark = pytest.mark.gpu


def say(*a):
    print(*a, flush=True)
    sys.stdout.flush()


@pytest.mark.parametrize("dims,spacing,drop,tfs", [
    ((7, 9, 8), 0.14, 0, 8),       # 504 particles, rows of up to ~500
    ((13, 13, 13), 0.12, 0, 8),    # rows of up to ~1,700: six rounds of masks
    ((9, 9, 9), 0.5, 300, 16),     # a drop of 0.14 in a body of ordinary spacing
    ((11, 12, 10), 0.32, 0, 16),   # rows on either side of 96
    ((8, 8, 8), 0.2, 0, 3),
])
def test_against_oracle(built, dims, spacing, drop, tfs):
    sc = with_drop(dims, 4, True, spacing, drop)
    for t in range(F.NUM_TF):
        sc.genome.tf_diffusability[t] = int(t >= F.NUM_TF - tfs)
    sc.buffers[F.FCONC][:] = np.random.default_rng(3).uniform(0, 1, (sc.n, F.NUM_TF))
    say("case: crowded diffusion", sc.n, "spacing", spacing, "drop", drop, "diffusing", tfs)
    g, o = pair(sc)
    for sim in (g, o):
        sim.Run2PhysicalSort()
        sim.step(3, sc.dt, sc.flags | (F.STEP_GRAPH if sim is g else 0))
    compare_all(g, o, "three steps")
    for sim in (g, o):
        sim.ComputeDiffusionCL()
    compare_all(g, o, "a diffusion pass")
    for sim in (g, o):
        sim.Run2GeneAction()
        sim.Run2PhysicalSort()
        sim.step(1, 1e-3, sc.flags)  # beyond the skin: the candidates are tested again
    compare_all(g, o, "gene action and a long step")


@pytest.mark.parametrize("dims,spacing,drop,most", [
    ((20, 20, 20), 0.14, 0, 5.0),      # 8.8 through the list of hits, 3.1 from masks
    ((64, 64, 64), 0.5, 3000, 3.0),    # 6.1 with later windows tested by the readers, 1.4 in rounds
])
def test_time_beside_the_pressure(built, dims, spacing, drop, most):
    sc = with_drop(dims, 6, True, spacing, drop)
    say("case: time of crowded diffusion", sc.n, "spacing", spacing, "drop", drop)
    sim = FluidSystem(sc.n, sc.b)
    sim.load_scene(sc)
    sim.Run2PhysicalSort()
    sim.step(2, 1e-6, sc.flags)
    best = {}
    for _ in range(4):
        ms, calls = (C.c_double * 12)(), (C.c_int * 12)()
        assert sim.lib.mg_step_timed(sim.h, 5, C.c_float(1e-6), sc.flags, ms, calls) == F.MG_OK
        for name, phase in (("pressure", 0), ("diffusion", 3)):
            best[name] = min(best.get(name, 1e9), ms[phase] / calls[phase])
    say("ms", best)
    assert best["diffusion"] < most * best["pressure"], best
    sim.close()
