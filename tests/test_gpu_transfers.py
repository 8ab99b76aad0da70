"""The boundary's copies through pinned halves (host_copy): what goes up comes down, byte for byte,
at the sizes where the path changes (4 MB to the host, 16 MB to the device, more helper threads
from 32 MB), at lengths that chunks and helpers do not divide, and for several handles from
several threads."""
import sys
import threading

import numpy as np
import pytest

from morphogenesis_amd import _ffi as F
from morphogenesis_amd import scenes

pytestmark = pytest.mark.gpu


def system(n, b=0):
    from morphogenesis_amd.fluid_system import FluidSystem

    sim = FluidSystem(n, b)
    sim.set_grid(scenes.make_grid((0, 0, 0), (8, 8, 8)))
    sim.set_params(scenes.make_params((0, 0, 0), (8, 8, 8)))
    return sim


def words(rng, shape, dtype):
    return rng.integers(0, 1 << 32, shape, dtype=np.uint64).astype(np.uint32).view(dtype)


# FCONC rows of 64 bytes: 64 B, 4 MB - 64, 4 MB, 4 MB + 64, 16 MB - 64, 16 MB, 16 MB + 64, 33 MB
@pytest.mark.parametrize("n", [1, 65535, 65536, 65537, 262143, 262144, 262145, 540673])
def test_round_trip(built, n):
    print("case: round trip", n * 64, "bytes", flush=True)
    sys.stdout.flush()
    sim = system(n)
    for seed in (1, 2):
        rng = np.random.default_rng(seed)
        conc = words(rng, (n, F.NUM_TF), np.float32)
        age = words(rng, (n,), np.uint32)
        sim.upload(F.FCONC, conc)
        sim.upload(F.FAGE, age)
        assert np.array_equal(sim.download(F.FCONC).view(np.uint32), conc.view(np.uint32))
        assert np.array_equal(sim.download(F.FAGE), age)
    sim.close()


def test_several_threads(built):
    bad = []

    def work(k):
        rng = np.random.default_rng(k)
        sim = system(270000 + 777 * k)
        for _ in range(4):
            conc = words(rng, (sim.n, F.NUM_TF), np.float32)
            sim.upload(F.FCONC, conc)
            if not np.array_equal(sim.download(F.FCONC).view(np.uint32), conc.view(np.uint32)):
                bad.append(k)
        sim.close()

    print("case: four threads, a handle each", flush=True)
    t = [threading.Thread(target=work, args=(k,)) for k in range(4)]
    for x in t:
        x.start()
    for x in t:
        x.join()
    assert not bad
