"""Dense groups split by rows in the fused steps of larger models (`dense_groups`) against the FP32
oracle, bit for bit: a drop of crowded cells beside a body of ordinary spacing, above the sizes at
which the diffusion, the force without bonds and the force with bonds go back to a lane per particle;
crowding throughout, which lists nothing and keeps the one-lane pressure; and a drop that is there
only after the homes were numbered. (The 4,194,304-particle configuration has more dense groups than
the list holds.)"""
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


def with_drop(dims, b, genes, spacing, drop, seed=7):
    """The tissue with its last `drop` particles in a cube of spacing 0.14 just above it."""
    sc = scenes.tissue(b=b, seed=seed, dims=dims, spacing=spacing, jitter=0.1 * spacing, genes=genes)
    rng = np.random.default_rng(seed)
    pos = sc.buffers[F.FPOS]
    if drop:
        side = int(np.ceil(drop ** (1 / 3)))
        cube = np.stack(np.meshgrid(*[np.arange(side)] * 3, indexing="ij"), -1).reshape(-1, 3)[:drop]
        mid = (pos[:, :3].min(0) + pos[:, :3].max(0)) / 2
        pos[-drop:, :3] = mid + 0.14 * (cube - side / 2) + rng.uniform(-0.01, 0.01, (drop, 3))
    for k in (F.FVEL, F.FVEVAL):
        sc.buffers[k][:, :3] = rng.normal(0.0, 2.0, (sc.n, 3))
    return sc


@pytest.mark.parametrize("dims,b,genes,sph,spacing,drop", [
    ((32, 32, 57), 6, True, 0, 0.5, 1000),   # 58,368: diffusion
    ((51, 51, 51), 0, False, 1, 0.5, 1000),  # 132,651: force without bonds
    ((48, 48, 65), 6, True, 0, 0.5, 3000),   # 149,760: force with bonds, diffusion
    ((41, 42, 41), 4, True, 0, 0.26, 0),     # 70,602: crowded throughout
])
def test_dense_groups_match_oracle(built, dims, b, genes, sph, spacing, drop):
    sc = with_drop(dims, b, genes, spacing, drop)
    say("case: dense", sc.n, "B", b, "genes", genes, "kernels", sph, "drop", drop)
    g, o = pair(sc)
    for sim in (g, o):
        sim.set_sph_kernels(sph)
        sim.Run2PhysicalSort()
        sim.step(3, sc.dt, sc.flags | (F.STEP_GRAPH if sim is g else 0))
    compare_all(g, o, "three steps")
    for sim in (g, o):
        sim.Run2InnerPhysicalLoop(sc.dt)
        sim.Run2GeneAction()
        sim.Run2PhysicalSort()
        sim.step(1, sc.dt, sc.flags)
    compare_all(g, o, "a loop and a step")


def test_drop_appears_and_goes(built):
    """The choice is made when the homes are numbered; positions change on either side of it."""
    plain, drop = (with_drop((32, 32, 57), 4, True, 0.5, d) for d in (0, 1000))
    g, o = pair(plain)
    for sim in (g, o):
        sim.Run2PhysicalSort()
        sim.step(2, plain.dt, plain.flags)
    for sc in (drop, plain):
        for sim in (g, o):
            sim.upload(F.FPOS, sc.buffers[F.FPOS])
            sim.Run2PhysicalSort()
            sim.step(2, sc.dt, sc.flags | (F.STEP_GRAPH if sim is g else 0))
        say("phase: positions replaced")
        compare_all(g, o, "positions replaced")
