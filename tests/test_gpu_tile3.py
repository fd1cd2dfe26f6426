"""In-wave y and z passes of the radix-3 lengths against the block passes
(FLUSI_TILE_WAVE=0): the same state to the round-off of their transforms."""
import os

import numpy as np
import pytest

import flusi_amd
from tests._util import GOLDEN, rel_l2, rewrite_ini

pytestmark = pytest.mark.gpu

# eps * log2(N) per transform, three steps, with a margin of about ten
TOL = {flusi_amd.FP64: 3e-14, flusi_amd.FP32_MIXED: 1.5e-5}
# one short y and z axis each, partial tiles (nx/2 + 1 = 9, 25 lines), both long
SHAPES = [(16, 96, 32), (16, 32, 96), (48, 192, 16), (32, 16, 192), (16, 384, 32), (16, 32, 384), (32, 96, 192)]


@pytest.mark.parametrize("prec", [flusi_amd.FP64, flusi_amd.FP32_MIXED])
@pytest.mark.parametrize("prune", ["0", "1"])
@pytest.mark.parametrize("shape", SHAPES)
def test_in_wave_radix3_tiles_match_block_tiles(tmp_path, monkeypatch, shape, prune, prec):
    ini = rewrite_ini(os.path.join(GOLDEN, "vortex_ring1_AB2", "vortexring1_AB2.ini"), str(tmp_path),
                      Resolution__nx=shape[0], Resolution__ny=shape[1], Resolution__nz=shape[2],
                      Time__dt_fixed="1.0e-3", Saving__itdrag="100000", Saving__tintegral="1.0e9", Saving__tsave="1.0e9")
    print(f"[tile3] {shape} {prune} {prec}", flush=True)
    monkeypatch.setenv("FLUSI_PRUNE", prune)
    rng = np.random.default_rng(2)
    f = rng.standard_normal((shape[2], shape[1], shape[0]))
    out = []
    for wave in ("1", "0"):
        monkeypatch.setenv("FLUSI_TILE_WAVE", wave)
        with flusi_amd.Flusi(ini, prec) as s:
            s.init_fields()
            s.set_uk(np.stack([s.fft(np.roll(f, i)) for i in range(3)]))
            s.advance(3)
            out.append((s.get_uk(), s.get_u(), s.fft(f)))
    for a, b in zip(*out):
        assert rel_l2(a, b) <= TOL[prec]
