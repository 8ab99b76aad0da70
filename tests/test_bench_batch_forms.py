"""bench.py's comparison of the batch's launch forms, on the CPU with a stand-in batch: each form is
timed under its own name, a form that the batch cannot take is left out, and the measured form is in
use again afterwards."""
import importlib
import os
import sys

import pytest

REPO = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))


class Stub:
    def __init__(self, form, can):
        self.now, self.can, self.stepped = form, can, []

    def form(self):
        return self.now

    def set_form(self, form):
        self.now = form if form in self.can else "dispatch"

    def step(self, n, dt, flags):
        self.stepped.append((self.now, n))

    def sync(self):
        pass


@pytest.mark.parametrize("form", ["merged", "persistent", "dispatch"])
@pytest.mark.parametrize("can", [("merged", "persistent", "dispatch"), ("merged", "dispatch")])
def test_forms_are_timed_under_their_names(form, can):
    sys.path.insert(0, REPO)
    bench = importlib.import_module("bench")
    if form not in can:
        pytest.skip("a form the batch cannot take is never in use")
    bat = Stub(form, can)
    got = bench.time_other_forms(bat, 7, 1e-4, 1, form, 1.25)
    assert set(got) == set(can) and got[form] == 1.25
    assert bat.form() == form
    assert {f for f, n in bat.stepped if n == 7} == set(can) - {form}
    assert set(bench.BATCH_STEP) == {"merged", "persistent", "dispatch"}
