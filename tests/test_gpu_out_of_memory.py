"""Device allocations that fail: the call reports it, or takes the route that needs no memory, and the
next call answers as if nothing had happened. The failure is a real one of the HIP runtime's (the
library asks for 2^60 bytes in place of one of its allocations, mg_debug_fail_allocation)."""
import sys

import numpy as np
import pytest

from morphogenesis_amd import _ffi as F
from morphogenesis_amd.fluid_system import FluidSystem
from tests.helpers import assert_bits_equal
from tests.test_gpu_dense import with_drop

pytestmark = pytest.mark.gpu


def say(*a):
    print(*a, flush=True)
    sys.stdout.flush()


@pytest.mark.parametrize("drop", [1000, 0])
def test_step_without_its_optional_buffers(built, drop):
    """A first step's list of dense groups, hit masks or bond records cannot be allocated: the step
    takes the route without them, and the one after it has them again."""
    sc = with_drop((32, 32, 57), 6, True, 0.5, drop)

    def run(fail):
        sim = FluidSystem(sc.n, sc.b)
        sim.load_scene(sc)
        sim.Run2PhysicalSort()
        sim.lib.mg_debug_fail_allocation(fail)
        sim.step(1, sc.dt, sc.flags)
        sim.lib.mg_debug_fail_allocation(0)
        sim.step(4, sc.dt, sc.flags | F.STEP_GRAPH)
        out = {buf: sim.download(buf) for buf in (F.FPOS, F.FVEL, F.FVEVAL, F.FPRESS, F.FDENSITY, F.FGCELL, F.FGNDX,
                                                  F.FCONC, F.FEPIGEN, F.FELASTIDX, F.FBIN_COUNT, F.FBIN_OFFSET)}
        sim.close()
        return out

    want = run(0)
    for k in (1, 2, 3):
        say("case: step of", sc.n, "with a drop of", drop, "allocation", k, "fails")
        got = run(k)
        for buf in want:
            assert_bits_equal(got[buf], want[buf], f"allocation {k} failed: {F.BUFFER_NAMES[buf]}")


def test_training_workspace(built):
    """Each of the training workspace's twelve allocations failing in turn, then the same gradients."""
    from morphogenesis_amd.learned import Net
    from tests.test_gpu_learned import identity_norm, random_data

    X, T, M = random_data(300, 4)

    def net():
        n = Net(seed=3)
        n.set_norm(*identity_norm(), 1.0)
        n.load_data(X, T, M)
        return n

    want = net()
    loss, g = want.grad(7, 290)
    want.close()
    for k in range(1, 13):
        say("case: training workspace, allocation", k, "fails")
        n = net()
        n.lib.mg_debug_fail_allocation(k)
        with pytest.raises(F.MgError):
            n.grad(7, 290)
        loss2, g2 = n.grad(7, 290)
        assert loss2 == loss and np.array_equal(g, g2), k
        n.close()
