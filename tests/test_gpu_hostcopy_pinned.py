"""Large copies from and to pinned host arrays: what goes in comes out."""
import ctypes

import numpy as np
import pytest
import torch

import flusi_amd
from tests._util import GOLDEN, rewrite_ini

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("prec", [flusi_amd.FP64, flusi_amd.FP32_MIXED])
def test_state_round_trip_of_pinned_arrays(tmp_path, prec):
    shape = (256, 128, 128)  # 202 MB of FP64
    ini = rewrite_ini(f"{GOLDEN}/vortex_ring1_AB2/vortexring1_AB2.ini", str(tmp_path), Resolution__nx=shape[0],
                      Resolution__ny=shape[1], Resolution__nz=shape[2])
    with flusi_amd.Flusi(ini, prec) as s:
        n = 6 * s.nxh * s.ny * s.nz
        a = torch.empty(n, dtype=torch.float64, pin_memory=True)
        a.copy_(torch.from_numpy(np.random.default_rng(2).standard_normal(n)))
        b = torch.zeros(n, dtype=torch.float64, pin_memory=True)
        p = lambda t: ctypes.cast(t.data_ptr(), ctypes.POINTER(ctypes.c_double))  # noqa: E731
        for _ in range(2):
            s._check(s._lib.flusi_set_uk(s._ctx, p(a)))
            s._check(s._lib.flusi_get_uk(s._ctx, p(b)))
        ref = a if prec == flusi_amd.FP64 else a.to(torch.float32).to(torch.float64)
        assert torch.equal(b, ref)
        assert np.array_equal(s.get_uk().view(np.float64).ravel(), ref.numpy())
