"""The autotuner times the passes that the configured stepper runs: pruned on
both sides (AB2, RK4), on one side (RK2), or not at all, and keeps its choice
for each of them."""
import os

import numpy as np
import pytest

import flusi_amd
from tests._util import GOLDEN, rewrite_ini

pytestmark = pytest.mark.gpu


def _ini(tmp_path, n, method):
    return rewrite_ini(os.path.join(GOLDEN, "vortex_ring1_AB2", "vortexring1_AB2.ini"), str(tmp_path),
                       name=f"{method}.ini", Resolution__nx=n, Resolution__ny=n, Resolution__nz=n,
                       Time__iTimeMethodFluid=method, Time__dt_fixed="1.0e-3", Saving__itdrag="100000",
                       Saving__tintegral="1.0e9", Saving__tsave="1.0e9")


@pytest.mark.parametrize("n", [48, 96, 128])
def test_methods_are_tuned_apart(tmp_path, n):
    """A choice cached for one method's passes is not taken for another's, and
    the state is left as it was."""
    ms = {}
    for method in ("RK2", "RK4", "AB2"):
        with flusi_amd.Flusi(_ini(tmp_path, n, method), flusi_amd.FP32_MIXED) as s:
            s.init_fields()
            s.advance(2)
            k = s.get_uk()
            v, ms[method] = s.autotune(reps=2)
            assert s.autotune(reps=2) == (v, ms[method])
            assert np.array_equal(s.get_uk(), k)
    assert len({ms[m] for m in ms}) == 3


def test_time_is_that_of_the_pruned_passes(tmp_path, monkeypatch):
    """At 256^3 an RK4 right-hand side without the modes outside the dealiased
    region takes about 0.6 of the time of one with every mode."""
    ms = {}
    for prune in ("0", "1"):
        monkeypatch.setenv("FLUSI_PRUNE", prune)
        with flusi_amd.Flusi(_ini(tmp_path, 256, "RK4"), flusi_amd.FP32_MIXED) as s:
            s.init_fields()
            s.advance(2)
            ms[prune] = s.autotune(reps=5)[1]
    assert ms["1"] < 0.85 * ms["0"]
