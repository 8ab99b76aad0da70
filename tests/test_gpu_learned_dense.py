"""Learned steps of models that list dense groups, above the sizes at which the force goes back to a
lane per particle (k_force_rows beside k_force): a zero network's steps equal the plain steps of the
same length, which the oracle's tests cover, and groups are listed."""
import ctypes as C
import sys

import numpy as np
import pytest

from morphogenesis_amd import _ffi as F
from morphogenesis_amd.fluid_system import FluidSystem
from tests.helpers import assert_bits_equal
from tests.test_gpu_dense import with_drop

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("dims,b", [((48, 48, 65), 6), ((51, 51, 51), 1), ((32, 32, 57), 6)])
def test_zero_network_is_the_plain_step(built, dims, b):
    from morphogenesis_amd.learned import Net

    sc = with_drop(dims, b, True, 0.5, 3000)
    print("case: learned steps with dense groups,", sc.n, "B", b, flush=True)
    sys.stdout.flush()
    net = Net(seed=1)
    net.set_params(np.zeros(net.nparams, np.float32))
    learned, plain = FluidSystem(sc.n, sc.b), FluidSystem(sc.n, sc.b)
    for sim in (learned, plain):
        sim.load_scene(sc)
        sim.Run2PhysicalSort()
    learned.step_learned(net, 3, 4 * sc.dt, sc.flags | F.STEP_GRAPH)
    plain.step(3, 4 * sc.dt, sc.flags)
    listed = C.c_uint32()
    assert learned.lib.mg_debug_crowding(learned.h, None, None, C.byref(listed)) == F.MG_OK
    assert listed.value > 0
    for buf in (F.FPOS, F.FVEL, F.FVEVAL, F.FCONC, F.FPRESS, F.FGCELL, F.FEPIGEN):
        a, c = learned.download(buf), plain.download(buf)
        assert np.array_equal(a, c), F.BUFFER_NAMES[buf]  # +0 == -0
    assert_bits_equal(learned.download(F.FELASTIDX), plain.download(F.FELASTIDX), "FELASTIDX")
    for sim in (learned, plain):
        sim.close()
    net.close()
