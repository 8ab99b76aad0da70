"""Particles at exactly one position with different velocities. They exert nothing on each other (a
zero distance is no hit), but the advance separates them, so in the same step they diffuse: the hit
masks of the pressure pass, which the diffusion visits, have to hold such pairs. Bit-equal to the
oracle in every form of the step: split by rows, a lane per particle (the crowded models' pressure,
and wide cells), and the batch's merged, dispatch and persistent forms."""
import ctypes as C
import sys

import numpy as np
import pytest

from morphogenesis_amd import _ffi as F
from morphogenesis_amd import scenes
from tests.helpers import assert_bits_equal
from tests.test_gpu_parity import compare_all, pair

pytestmark = pytest.mark.gpu


def say(*a):
    print(*a, flush=True)
    sys.stdout.flush()


def paired(dims, b, spacing, seed=11, pairs=200):
    """A tissue whose first particles sit in pairs at one position, without bonds of their own."""
    sc = scenes.tissue(b=b, seed=seed, dims=dims, spacing=spacing, jitter=0.1 * spacing, genes=True)
    rng = np.random.default_rng(seed)
    at = rng.choice(sc.n, (min(pairs, sc.n // 4), 2), replace=False)
    pos, rec = sc.buffers[F.FPOS], sc.buffers[F.FELASTIDX]
    pos[at[:, 0]] = pos[at[:, 1]]
    gone = np.isin(rec[:, :, 0], at)
    gone[at.reshape(-1)] = True
    rec[gone] = 0
    rec[gone, 0] = rec[gone, 5] = F.NONE
    sc.buffers[F.FCONC][:] = rng.uniform(0, 1, (sc.n, F.NUM_TF))
    for k in (F.FVEL, F.FVEVAL):
        sc.buffers[k][:, :3] = rng.normal(0.0, 2.0, (sc.n, 3))
    return sc


@pytest.mark.parametrize("dims,b,spacing,sph", [
    ((8, 8, 8), 4, 0.5, 0),        # nine wavefronts per 64 particles
    ((55, 56, 57), 4, 0.28, 0),    # 175,560 crowded throughout: the pressure a lane per particle
    ((55, 56, 57), 0, 0.28, 1),
    ((40, 40, 40), 4, 0.5, 0),     # three wavefronts
])
def test_single_model(built, dims, b, spacing, sph):
    sc = paired(dims, b, spacing)
    say("case: coincident pairs", sc.n, "B", b, "spacing", spacing, "kernels", sph)
    g, o = pair(sc)
    for sim in (g, o):
        sim.set_sph_kernels(sph)
        sim.Run2PhysicalSort()
        sim.step(1, sc.dt, sc.flags)
    crowded = C.c_int()
    assert g.lib.mg_debug_crowding(g.h, None, C.byref(crowded), None) == F.MG_OK
    assert crowded.value == int(sc.n > 163840)
    compare_all(g, o, "one step")
    for sim in (g, o):
        sim.step(2, sc.dt, sc.flags | (F.STEP_GRAPH if sim is g else 0))
    compare_all(g, o, "three steps")


@pytest.mark.parametrize("form", ["merged", "dispatch", "persistent"])
def test_batch_forms(built, form):
    from morphogenesis_amd.batch import Batch

    scs = [paired(d, 4, s, seed=20 + k) for k, (d, s) in enumerate([((5, 5, 6), 0.5), ((12, 11, 13), 0.3)])]
    say("case: coincident pairs, batch", form, [sc.n for sc in scs])
    both = [pair(sc) for sc in scs]
    for g, o in both:
        g.Run2PhysicalSort()
        o.Run2PhysicalSort()
    bat = Batch([g for g, _ in both])
    if form != "merged":
        bat.set_persistent(form == "persistent")
    bat.step(1, scs[0].dt, F.STEP_GENES)
    bat.step(2, scs[0].dt, F.STEP_GENES | F.STEP_GRAPH)
    bat.sync()
    for k, (g, o) in enumerate(both):
        o.step(3, scs[0].dt, F.STEP_GENES)
        for buf in (F.FPOS, F.FVEL, F.FPRESS, F.FCONC, F.FEPIGEN, F.FGCELL):
            assert_bits_equal(g.download(buf), o.download(buf), f"instance {k}: {F.BUFFER_NAMES[buf]}")
    bat.close()
