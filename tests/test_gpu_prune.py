"""Steps whose passes skip the modes outside the dealiased region against the
same steps with every mode moved and transformed (FLUSI_PRUNE=0): the same
sums without their zero terms, so the states agree to round-off."""
import os

import numpy as np
import pytest

import flusi_amd
from tests._util import CONFIGS, GOLDEN, rel_l2, rewrite_ini

pytestmark = pytest.mark.gpu

# a few transforms' round-off per step: eps * log2(N) with a margin of about ten
TOL = {flusi_amd.FP64: 1e-14, flusi_amd.FP32_MIXED: 4e-6}


def _ini(tmp_path, shape, method, sponge, fixed_mean):
    nx, ny, nz = shape
    kw = dict(Resolution__nx=nx, Resolution__ny=ny, Resolution__nz=nz, Time__iTimeMethodFluid=method,
              Time__dt_fixed="1.0e-3", Saving__itdrag="100000", Saving__tintegral="1.0e9", Saving__tsave="1.0e9")
    src = os.path.join(GOLDEN, "vortex_ring1_AB2", "vortexring1_AB2.ini")
    if sponge:
        kw.update(Sponge__iVorticitySponge="yes", Sponge__iSpongeType="cavity", Sponge__eps_sponge="0.1",
                  Sponge__sponge_thickness="3")
    if fixed_mean:
        kw.update(MeanFlow__iMeanFlow_x="fixed", MeanFlow__ux="0.7")
    return rewrite_ini(src, str(tmp_path), **kw)


def _run(ini, prec, uk0, steps):
    with flusi_amd.Flusi(ini, prec) as s:
        s.init_fields()
        if uk0 is not None:
            s.set_uk(uk0)
        s.advance(steps)
        return s.get_uk(), s.get_u(), s.energy_k()


# radix-3 and power-of-two axes, the smallest, lines that fill a tile exactly
# (2 ym + 1 = 63) and that leave one position over, one axis of 512
SHAPES = [(16, 16, 16), (32, 24, 48), (96, 64, 32), (64, 96, 128), (48, 128, 192), (16, 512, 64), (512, 16, 32),
          (32, 64, 512), (192, 32, 16), (256, 16, 384)]


@pytest.mark.parametrize("prec", [flusi_amd.FP64, flusi_amd.FP32_MIXED])
@pytest.mark.parametrize("method", ["AB2", "RK2", "RK4"])
@pytest.mark.parametrize("shape", SHAPES)
def test_pruned_steps_match_full_steps(tmp_path, monkeypatch, shape, method, prec):
    """Three steps from a state with modes outside the region (the first step
    is then not pruned), through set_uk."""
    nx, ny, nz = shape
    ini = _ini(tmp_path, shape, method, sponge=shape[0] == 96, fixed_mean=shape[0] == 32)
    print(f"[prune] {shape} {method} {prec}", flush=True)
    rng = np.random.default_rng(3)
    with flusi_amd.Flusi(ini, flusi_amd.FP64) as s:
        s.init_fields()
        uk0 = np.stack([s.fft(rng.standard_normal((nz, ny, nx))) for _ in range(3)])
    monkeypatch.setenv("FLUSI_PRUNE", "1")  # below the sizes where it pays, too
    uk, u, e = _run(ini, prec, uk0, 3)
    monkeypatch.setenv("FLUSI_PRUNE", "0")
    uk_f, u_f, e_f = _run(ini, prec, uk0, 3)
    assert rel_l2(uk, uk_f) <= TOL[prec]
    assert rel_l2(u, u_f) <= TOL[prec]
    assert abs(e - e_f) <= TOL[prec] * e_f
    if method != "RK2":  # outside the region: zero
        assert np.array_equal(uk == 0, uk_f == 0)


@pytest.mark.parametrize("prec", [flusi_amd.FP64, flusi_amd.FP32_MIXED])
def test_pruned_insect_run_and_restart_of_the_state(tmp_path, monkeypatch, prec):
    """From rest (pruned from the first stage), then a state with modes outside
    the region set into the running context, then on."""
    n = 64
    ini = rewrite_ini(os.path.join(CONFIGS, "cfg3_insect_512.ini"), str(tmp_path), Resolution__nx=n, Resolution__ny=n,
                      Resolution__nz=n, Time__dt_fixed="2.0e-4")
    rng = np.random.default_rng(5)

    def run():
        with flusi_amd.Flusi(ini, prec) as s:
            s.init_fields()
            s.advance(2)
            a = s.get_u()
            s.set_uk(s.get_uk() + 1e-3 * np.stack([s.fft(rng.standard_normal((n, n, n))) for _ in range(3)]))
            s.advance(2)
            return a, s.get_u()

    a, b = run()
    monkeypatch.setenv("FLUSI_PRUNE", "0")
    rng = np.random.default_rng(5)
    a_f, b_f = run()
    assert rel_l2(a, a_f) <= TOL[prec]
    assert rel_l2(b, b_f) <= TOL[prec]
