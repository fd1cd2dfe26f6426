"""The x pass with pairs of lines in one transform against the block x pass
(FLUSI_XWAVE=0): the same right-hand side to the round-off of its transforms."""
import os

import pytest

import flusi_amd
from tests._util import CONFIGS, rel_l2, rewrite_ini

pytestmark = pytest.mark.gpu

# eps * log2(N) of three transforms, with a margin of about ten
TOL = {flusi_amd.FP64: 3e-14, flusi_amd.FP32_MIXED: 1.5e-5}
# every length; few lines (one wave a block, four positions a lane), lines that
# leave a wave's last pairs empty (16 x 24 = 384 lines), many lines
SHAPES = [(n, 16, 16) for n in (32, 48, 64, 96, 128, 192, 256, 384, 512)] + \
    [(32, 24, 16), (48, 24, 16), (96, 24, 16), (64, 128, 128), (96, 96, 128), (128, 96, 96), (256, 64, 64)]


@pytest.mark.parametrize("prec", [flusi_amd.FP64, flusi_amd.FP32_MIXED])
@pytest.mark.parametrize("sponge", ["no", "cavity", "outlet_x"])
@pytest.mark.parametrize("shape", SHAPES)
def test_pair_x_pass_matches_block_x_pass(tmp_path, monkeypatch, shape, sponge, prec):
    """N(u) (undealiased input), then two adaptive steps of a dealiased state,
    which use the statistics, the pruned input and the mask flags."""
    nx, ny, nz = shape
    h = 2.0 / min(ny, nz)
    ini = rewrite_ini(os.path.join(CONFIGS, "cfg2_sphere_256x128x128.ini"), str(tmp_path), Resolution__nx=nx,
                      Resolution__ny=ny, Resolution__nz=nz, Geometry__xl=repr(nx * h), Geometry__yl=repr(ny * h),
                      Geometry__zl=repr(nz * h), Geometry__x0=repr(0.4 * nx * h), Geometry__y0=repr(0.5 * ny * h),
                      Geometry__z0=repr(0.5 * nz * h), Time__iTimeMethodFluid="AB2",
                      Sponge__iVorticitySponge="no" if sponge == "no" else "yes",
                      Sponge__iSpongeType="cavity" if sponge == "no" else sponge, Sponge__sponge_thickness=3,
                      Saving__tintegral=100.0, Saving__itdrag=100000)
    monkeypatch.setenv("FLUSI_PRUNE", "1")
    print(f"[xpair] {shape} {sponge} {prec}", flush=True)
    out = []
    for wave in ("1", "0"):
        monkeypatch.setenv("FLUSI_XWAVE", wave)
        with flusi_amd.Flusi(ini, prec) as s:
            s.init_fields()
            s.advance(3)
            n = s.cal_nlk(0.0)
            out.append((s.get_uk(), n, s.get_time()[3]))
    (u1, n1, dt1), (u0, n0, dt0) = out
    assert abs(dt1 - dt0) <= 1e-12 * dt0
    assert rel_l2(u1, u0) <= TOL[prec]
    assert rel_l2(n1, n0) <= TOL[prec]
