"""What a captured step of an ensemble replays: its passes, and not the
clearing of registers that its first pruned step needs once."""
import os
import time

import pytest

import flusi_amd
from tests._util import GOLDEN, rewrite_ini

pytestmark = pytest.mark.gpu


def _step_us(tmp_path, inicond):
    n, members, steps = 128, 4, 30
    inis = [rewrite_ini(os.path.join(GOLDEN, "vortex_ring1_AB2", "vortexring1_AB2.ini"), str(tmp_path), name=f"{inicond}{i}.ini",
                        Resolution__nx=n, Resolution__ny=n, Resolution__nz=n, Time__iTimeMethodFluid="RK4",
                        Time__dt_fixed="1.0e-3", InitialCondition__inicond=inicond, Saving__itdrag="100000",
                        Saving__tintegral="1.0e9", Saving__tsave="1.0e9") for i in range(members)]
    best = float("inf")
    with flusi_amd.Ensemble(inis, flusi_amd.FP32_MIXED) as e:
        e.init_fields()
        e.advance(10, flusi_amd.ENSEMBLE_GRAPH)
        for _ in range(6):
            t = time.perf_counter()
            e.advance(steps, flusi_amd.ENSEMBLE_GRAPH)
            best = min(best, (time.perf_counter() - t) / steps * 1e6)
    return best


def test_registers_are_not_cleared_in_every_replay(tmp_path):
    """From a vortex ring the first RK4 step is not pruned and leaves modes
    outside the dealiased region in both registers; from rest it leaves none.
    The replayed steps do the same work (clearing both took 16 % more)."""
    assert _step_us(tmp_path, "VortexRing") < 1.1 * _step_us(tmp_path, "quiescent")
