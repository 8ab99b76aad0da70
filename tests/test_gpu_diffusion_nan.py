"""A diffusion weight that is itself NaN (simulation scale 0: an infinite cut-off times zero) reaches
the concentrations, in the diffusion split by rows as in the oracle: a NaN is no mark of a candidate
that is not a hit."""
import sys

import numpy as np
import pytest

from morphogenesis_amd import _ffi as F
from morphogenesis_amd import scenes
from tests.test_gpu_parity import pair

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("fused", [True, False])
def test_nan_weights(built, fused):
    sc = scenes.tissue(n_side=8, b=4, seed=2)
    sc.buffers[F.FCONC][:] = np.random.default_rng(2).uniform(0, 1, (sc.n, F.NUM_TF))
    print("case: NaN diffusion weights, fused", fused, flush=True)
    sys.stdout.flush()
    got = []
    for sim in pair(sc):
        sim.Run2PhysicalSort()
        p = sc.params
        p.psimscale = 0.0
        sim.set_params(p)
        if fused:
            sim.step(1, sc.dt, F.STEP_GENES)
        else:
            sim.ComputeDiffusionCL()
        got.append(np.isnan(sim.download(F.FCONC)))
    assert got[1].any()
    assert np.array_equal(got[0], got[1]), (got[0].sum(), got[1].sum())
