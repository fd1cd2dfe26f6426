"""Copies of fields between host arrays and the device: what goes in comes out,
for plain copies and for chunks in threads (from 48 MB on), the last one with a
remainder."""
import threading

import numpy as np
import pytest

import flusi_amd
from tests._util import GOLDEN, rewrite_ini

pytestmark = pytest.mark.gpu


def _ini(tmp_path, shape):
    return rewrite_ini(f"{GOLDEN}/vortex_ring1_AB2/vortexring1_AB2.ini", str(tmp_path), Resolution__nx=shape[0],
                       Resolution__ny=shape[1], Resolution__nz=shape[2])


def _round_trip(ini, prec, seed, out=None):
    with flusi_amd.Flusi(ini, prec) as s:
        rng = np.random.default_rng(seed)
        a = rng.standard_normal((2,) + (s.nxh * s.ny * s.nz * 3,)).view(np.complex128).reshape(s.spectral_shape)
        for _ in range(2):
            s.set_uk(a)
            b = s.get_uk()
        ref = a if prec == flusi_amd.FP64 else a.astype(np.complex64).astype(np.complex128)
        ok = np.array_equal(b, ref)
        if out is not None:
            out.append(ok)
        return ok


@pytest.mark.parametrize("prec", [flusi_amd.FP64, flusi_amd.FP32_MIXED])
@pytest.mark.parametrize("shape", [(16, 16, 16), (128, 96, 64), (192, 128, 96), (256, 128, 128), (256, 96, 128), (512, 128, 128)])
def test_state_round_trip(tmp_path, shape, prec):
    print(f"[hostcopy] {shape} {prec}", flush=True)
    assert _round_trip(_ini(tmp_path, shape), prec, 1)


def test_state_round_trips_in_threads(tmp_path):
    """Contexts of several threads share the staging pool."""
    ini = _ini(tmp_path, (256, 128, 128))
    ok = []
    t = [threading.Thread(target=_round_trip, args=(ini, p, i, ok)) for i, p in
         enumerate([flusi_amd.FP64, flusi_amd.FP32_MIXED, flusi_amd.FP64])]
    for x in t:
        x.start()
    for x in t:
        x.join()
    assert ok == [True, True, True]
