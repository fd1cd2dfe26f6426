"""The mask's line flags where no mask is drawn: they stay valid, and a call
that draws nothing launches nothing."""
import os
import time

import numpy as np
import pytest

import flusi_amd
from tests._util import CONFIGS, GOLDEN, rewrite_ini

pytestmark = pytest.mark.gpu


def test_create_mask_without_penalization(tmp_path):
    """0.5 us a call (3.3 us with the launch of the flags' kernel)."""
    ini = rewrite_ini(os.path.join(GOLDEN, "vortex_ring1_AB2", "vortexring1_AB2.ini"), str(tmp_path), Resolution__nx=32,
                      Resolution__ny=32, Resolution__nz=32, Time__dt_fixed="1.0e-3")
    with flusi_amd.Flusi(ini, flusi_amd.FP64) as s:
        s.init_fields()
        s.create_mask(0.0)
        best = float("inf")
        for _ in range(20):
            t = time.perf_counter()
            for _ in range(50):
                s.create_mask(0.0)
            best = min(best, (time.perf_counter() - t) / 50 * 1e6)
        s.advance(2)
        u = s.get_u()
    assert best < 2.0
    with flusi_amd.Flusi(ini, flusi_amd.FP64) as s:
        s.init_fields()
        s.advance(2)
        assert np.array_equal(s.get_u(), u)


def test_create_mask_redraws_a_resting_mask(tmp_path):
    """The flags after it are those of the mask: the same steps as without them."""
    ini = rewrite_ini(os.path.join(CONFIGS, "cfg2_sphere_256x128x128.ini"), str(tmp_path), Resolution__nx=64,
                      Resolution__ny=32, Resolution__nz=32, Time__dt_fixed="5.0e-4", Saving__tintegral=100.0,
                      Saving__itdrag=100000)
    out = []
    for again in (False, True):
        with flusi_amd.Flusi(ini, flusi_amd.FP64) as s:
            s.init_fields()
            s.advance(2)
            if again:
                s.create_mask(0.0)
            s.advance(2)
            out.append(s.get_u())
    assert np.array_equal(*out)
