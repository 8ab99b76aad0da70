"""bench.py names the kernels that a workload runs, on the CPU: the sweeps split by rows, a lane per
particle, and the insert without gene action, at sizes on either side of the library's (read from its
source)."""
import importlib
import os
import re
import sys
import types

import pytest

REPO = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))


@pytest.fixture(scope="module")
def bench():
    sys.path.insert(0, REPO)
    return importlib.import_module("bench")


def sizes():
    text = open(os.path.join(REPO, "morphogenesis_amd", "csrc", "mg_capi.hip")).read()
    return {k: int(re.search(r"\b%s = (\d+)" % k, text).group(1))
            for k in ("kForceRows9", "kForceRows3NoBonds", "kDiffuseRows")}


def scene(n, b=32, genes=True, srch=3, r2=1.0):
    ns = types.SimpleNamespace
    return ns(n=n, b=b, flags=int(genes), grid=ns(srch=srch), params=ns(r2=r2))


def test_names_follow_the_librarys_sizes(bench):
    k = sizes()
    for b, size in ((32, k["kForceRows9"]), (0, k["kForceRows3NoBonds"])):
        assert bench.kernels_of_phase(scene(size, b))["force"] == "k_force_advance_rows"
        assert bench.kernels_of_phase(scene(size + 1, b))["force"] == "k_force_advance"
    assert bench.kernels_of_phase(scene(k["kDiffuseRows"]))["diffusion"] == "k_diffuse_rows"
    assert bench.kernels_of_phase(scene(k["kDiffuseRows"] + 1))["diffusion"] == "k_diffuse_genes_insert"
    assert bench.kernels_of_phase(scene(1000, genes=False))["diffusion"] == "k_insert_next"
    for n in (1000, 262144):
        assert bench.kernels_of_phase(scene(n))["pressure"] == "k_pressure_rows"
    assert bench.kernels_of_phase(scene(262144), crowded=True)["pressure"] == "k_pressure"
    two = bench.kernels_of_phase(scene(1000, srch=2))
    assert (two["pressure"], two["force"], two["diffusion"]) == ("k_pressure", "k_force_advance", "k_diffuse_genes_insert")
