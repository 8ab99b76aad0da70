"""The batch's launch form as the program sees and sets it: by size, chosen, after the autotuner, and
after an autotuner that failed; and every instance bit-equal to one stepped alone in each of them, with
and without gene action."""
import sys

import numpy as np
import pytest

from morphogenesis_amd import _ffi as F
from morphogenesis_amd import scenes
from tests.helpers import assert_bits_equal
from tests.test_gpu_batch_merged import STATE, open_scene

pytestmark = pytest.mark.gpu

UPLOAD = [F.FPOS, F.FVEL, F.FVEVAL, F.FCONC, F.FEPIGEN, F.FELASTIDX, F.FPARTICLE_ID]


def say(*a):
    print(*a, flush=True)
    sys.stdout.flush()


def same_state(to, of):
    """`to` in the sorted state of `of`: the same particles in the same slots and homes."""
    for sim in (to, of):
        sim.Run2PhysicalSort()
    for buf in UPLOAD:
        x = of.download(buf)
        for sim in (to, of):
            sim.upload(buf, x)
    for sim in (to, of):
        sim.Run2PhysicalSort()


@pytest.mark.parametrize("genes", [True, False])
def test_forms(built, genes):
    from morphogenesis_amd.batch import Batch

    scs = [scenes.tissue(b=b, seed=60 + k, dims=d) for k, (d, b) in
           enumerate([((7, 8, 9), 6), ((20, 21, 22), 32), ((5, 5, 5), 4)])]
    for sc in scs:
        sc.buffers[F.FVEL][:, :3] = np.random.default_rng(sc.n).normal(0, 2.0, (sc.n, 3))
    say("case: batch forms", [sc.n for sc in scs], "genes", genes)
    together, alone = [open_scene(sc) for sc in scs], [open_scene(sc) for sc in scs]
    bat = Batch(together)
    flags = F.STEP_GENES if genes else 0
    dt = scs[0].dt

    def check(what, expect):
        assert bat.form() == expect, what
        bat.step(3, dt, flags | F.STEP_GRAPH)
        bat.step(2, dt, flags | F.STEP_GRAPH)
        assert bat.form() == expect, what
        assert bat.launch_config()[0] == int(expect == "persistent"), what
        bat.sync()
        for k, sim in enumerate(alone):
            sim.step(5, dt, flags)
            for buf in STATE:
                assert_bits_equal(together[k].download(buf), sim.download(buf), f"{what}, instance {k}: {F.BUFFER_NAMES[buf]}")

    check("by size", "merged")
    for form in ("persistent", "dispatch", "merged", "dispatch"):
        bat.set_form(form)
        check(form, form)
    bat.set_form("by size")
    check("by size again", "merged")
    bat.set_persistent(False)
    check("set_persistent(False)", "dispatch")
    bat.autotune(1, dt, flags)
    kept = bat.form()
    say("the autotuner keeps", kept)
    for a, b in zip(together, alone):  # its steps were real ones
        same_state(a, b)
    check("autotuned", kept)
    bat.set_form("by size")
    bat.lib.mg_debug_fail_allocation(5)
    with pytest.raises(F.MgError):
        bat.autotune(1, dt, flags)
    bat.lib.mg_debug_fail_allocation(0)
    for a, b in zip(together, alone):
        same_state(a, b)
    check("after an autotuner that failed", "merged")
    bat.close()
