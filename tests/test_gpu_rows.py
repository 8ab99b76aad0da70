"""The sweeps split by rows (nine or three wavefronts per 64 particles, `launch_pressure`,
`launch_force_advance`, `launch_diffuse_rows`) against the FP32 oracle, bit for bit, at the sizes
where they can go wrong: workgroups of one, 63, 64 and 65 particles; cells so full that a row has
more than 64 candidates, a wavefront's band exceeds its stage and a particle's hit list takes
several rounds; particles with more incoming bonds than the force keeps in registers; and both
sides of each size at which the split changes."""
import sys

import numpy as np
import pytest

from morphogenesis_amd import _ffi as F
from morphogenesis_amd import scenes
from tests.test_gpu_parity import compare_all, pair

pytestmark = pytest.mark.gpu


def say(*a):
    print(*a, flush=True)
    sys.stdout.flush()


def scene(dims, b, genes=True, spacing=0.5, drift=0.0, seed=5):
    sc = scenes.tissue(b=b, seed=seed, dims=dims, spacing=spacing, jitter=0.1 * spacing, genes=genes)
    if drift:
        for k in (F.FVEL, F.FVEVAL):
            sc.buffers[k][:, :3] = np.random.default_rng(seed).normal(0.0, drift, (sc.n, 3)).astype(np.float32)
    return sc


@pytest.mark.parametrize("dims,b,genes,spacing,drift,steps", [
    ((1, 1, 1), 4, True, 0.5, 0.0, 4),
    ((3, 3, 7), 4, True, 0.5, 5.0, 8),        # 63
    ((4, 4, 4), 32, True, 0.5, 5.0, 8),       # 64
    ((5, 13, 1), 0, False, 0.5, 5.0, 8),      # 65, no bonds
    ((9, 10, 11), 6, True, 0.22, 0.0, 6),     # ~94 particles per cell: wide rows, unstaged bands
    ((9, 9, 9), 32, True, 0.3, 50.0, 6),      # fast: diffusion tests its candidates itself
    ((10, 10, 10), 0, False, 0.22, 50.0, 6),
])
def test_small_models_match_oracle(built, dims, b, genes, spacing, drift, steps):
    sc = scene(dims, b, genes, spacing, drift)
    say("case: rows", sc.n, "B", b, "genes", genes, "spacing", spacing, "drift", drift)
    g, o = pair(sc)
    for sim in (g, o):
        sim.Run2PhysicalSort()
        sim.step(steps, sc.dt, sc.flags | (F.STEP_GRAPH if sim is g else 0))
    compare_all(g, o, "fused steps")
    say("phase: the loop of phase calls")
    for sim in (g, o):
        for _ in range(2):
            sim.Run2InnerPhysicalLoop(sc.dt)
            sim.Run2GeneAction()
            sim.Run2PhysicalSort()
    compare_all(g, o, "phase loop")


def test_many_incoming_bonds(built):
    """Every particle of a block bonded to by up to 40 others (dense lattice, wide bond radius)."""
    sc = scene((8, 8, 8), 64, True, 0.25, 1.0)
    rec = sc.buffers[F.FELASTIDX]
    rng = np.random.default_rng(3)
    for k in range(20, 64):  # random partners within the block in the free slots
        to = rng.integers(0, sc.n, sc.n)
        free = (rec[:, k, 0] == F.NONE) & (to != np.arange(sc.n))
        rec[free, k] = rec[free, 0]
        rec[free, k, 0] = to[free]
        rec[free, k, 5] = to[free] + 1
    say("case: incoming bonds", int((rec[:, :, 0] != F.NONE).sum()) / sc.n, "per particle")
    g, o = pair(sc)
    for sim in (g, o):
        sim.Run2PhysicalSort()
        sim.step(6, sc.dt, sc.flags)
    compare_all(g, o, "many incoming bonds")


@pytest.mark.parametrize("dims,b,genes,sph", [
    ((32, 32, 40), 0, False, 0), ((32, 32, 41), 0, False, 1),   # force without bonds: nine, three
    ((32, 32, 48), 6, True, 0), ((32, 32, 49), 6, True, 1),     # pressure: nine, three
    ((32, 32, 56), 6, True, 0), ((32, 32, 57), 6, True, 0),     # diffusion: by rows, a lane each
    ((48, 48, 56), 0, False, 0), ((48, 48, 57), 0, False, 0),   # force without bonds: three, a lane each
    ((48, 48, 64), 6, True, 0), ((48, 48, 65), 6, True, 0),     # force with bonds: nine, a lane each
])
def test_both_sides_of_each_size(built, dims, b, genes, sph):
    sc = scene(dims, b, genes, 0.5, 3.0)
    say("case: size", sc.n, "B", b, "kernels", sph)
    g, o = pair(sc)
    for sim in (g, o):
        sim.set_sph_kernels(sph)
        sim.Run2PhysicalSort()
        sim.step(2, sc.dt, sc.flags)
    compare_all(g, o, "two steps")
