"""A learned step given up between its passes, in a model whose steps list dense groups: an error of
the HIP runtime that the program left unread is found at the network's launch, the step returns it, and
the next step starts its list anew."""
import ctypes as C
import sys

import numpy as np
import pytest

from morphogenesis_amd import _ffi as F
from morphogenesis_amd.fluid_system import FluidSystem
from tests.helpers import assert_bits_equal
from tests.test_gpu_dense import with_drop
from tests.test_zz_no_alloc import hip_runtime

pytestmark = pytest.mark.gpu


def test_step_given_up_at_the_network(built):
    from morphogenesis_amd.learned import Net

    sc = with_drop((32, 32, 57), 6, True, 0.5, 1000)
    print("case: learned step given up,", sc.n, "with a drop", flush=True)
    sys.stdout.flush()
    hip = hip_runtime()
    net = Net(seed=1)
    net.set_params(np.zeros(net.nparams, np.float32))
    sims = []
    for give_up in (False, True):
        sim = FluidSystem(sc.n, sc.b)
        sim.load_scene(sc)
        sim.Run2PhysicalSort()
        sim.step_learned(net, 2, sc.dt, sc.flags)
        if give_up:
            p = C.c_void_p()
            assert hip.hipMalloc(C.byref(p), C.c_size_t(1 << 60)) != 0  # the error is left unread
            with pytest.raises(F.MgError):
                sim.step_learned(net, 1, sc.dt, sc.flags)
        sim.step_learned(net, 3, sc.dt, sc.flags)
        sims.append(sim)
    # (the bonds' integrators count the force pass of the step given up, too)
    for buf in (F.FPOS, F.FVEL, F.FVEVAL, F.FPRESS, F.FDENSITY, F.FGCELL, F.FGNDX, F.FCONC, F.FEPIGEN, F.FBIN_COUNT,
                F.FBIN_OFFSET):
        assert_bits_equal(sims[1].download(buf), sims[0].download(buf), F.BUFFER_NAMES[buf])
    for sim in sims:
        sim.close()
    net.close()
