"""The penalisation sums of the x pass (a dynamic mean flow, which takes them
into the zero mode) with pairs of lines in one transform, against the block x
pass (FLUSI_XWAVE=0): at nx = 96 below 2^20 points a pair takes 24 lanes, and
the 16 lanes a wave has over must not reach the sums, whatever an earlier
kernel left in LDS."""
import os

import numpy as np
import pytest

import flusi_amd
from tests._util import CONFIGS, GOLDEN, rel_l2, rewrite_ini

pytestmark = pytest.mark.gpu

# eps * log2(N) of three transforms, with a margin of about ten: per three
# right-hand sides, whose errors add at most linearly
TOL = {flusi_amd.FP64: 3e-14, flusi_amd.FP32_MIXED: 1.5e-5}
STAGES = {"AB2": 1, "RK2": 2, "RK4": 4}
EPS, M_FLUID, STEPS = 1.0e-3, 20.0, 3


def _sphere(tmp_path, name, shape, method, sponge, x0=0.4):
    nx, ny, nz = shape
    h = 2.0 / min(ny, nz)
    return rewrite_ini(os.path.join(CONFIGS, "cfg2_sphere_256x128x128.ini"), str(tmp_path), name=name, Resolution__nx=nx,
                       Resolution__ny=ny, Resolution__nz=nz, Geometry__xl=repr(nx * h), Geometry__yl=repr(ny * h),
                       Geometry__zl=repr(nz * h), Geometry__x0=repr(x0 * nx * h), Geometry__y0=repr(0.5 * ny * h),
                       Geometry__z0=repr(0.5 * nz * h), Geometry__Size="0.9", Penalization__eps=repr(EPS),
                       Time__iTimeMethodFluid=method, Time__dt_fixed="5.0e-4",
                       Sponge__iVorticitySponge="no" if sponge == "no" else "yes",
                       Sponge__iSpongeType="cavity" if sponge == "no" else sponge, Sponge__sponge_thickness=3,
                       MeanFlow__iMeanFlow_x="dynamic", MeanFlow__m_fluid=repr(M_FLUID), MeanFlow__uy="0.2",
                       MeanFlow__uz="-0.1", Saving__tintegral=100.0, Saving__itdrag=100000)


def _fill_lds(tmp_path):
    """Kernels whose workgroups together hold every compute unit's LDS, on a
    state of NaN: what they leave there is NaN."""
    ini = rewrite_ini(os.path.join(GOLDEN, "vortex_ring1_AB2", "vortexring1_AB2.ini"), str(tmp_path), name="fill.ini",
                      Resolution__nx=64, Resolution__ny=512, Resolution__nz=64)
    with flusi_amd.Flusi(ini, flusi_amd.FP64) as s:
        s.init_fields()
        s.set_uk(np.full(s.spectral_shape, complex(np.nan, np.nan)))
        s.cal_nlk(0.0)


def _check(s1, s0, prec, rhs):
    """(nlk, uk, u) of a run against the block x pass's."""
    (n1, k1, u1, mask), (n0, k0, u0, _) = s1, s0
    for a in (n1, k1, u1):
        assert np.all(np.isfinite(a))
    tol = TOL[prec] * max(1, rhs / 3)
    # -sum(mask/eps (u - us)) dV / m_fluid: no larger than with |u| = max|u|
    # everywhere, to which the velocity's error is relative
    dv = (2.0 / min(u0.shape[2], u0.shape[1])) ** 3
    scale = mask.sum() / EPS * dv / M_FLUID * np.max(np.abs(u0))
    assert abs(n0[0, 0, 0, 0].real) > 1e-3 * scale  # (the sphere stands in a flow along x)
    assert np.max(np.abs(n1[0, 0, 0, 0] - n0[0, 0, 0, 0])) <= tol * scale
    assert np.max(np.abs(k1[:, 0, 0, 0] - k0[:, 0, 0, 0])) <= tol * np.max(np.abs(u0))
    for a, b in ((n1, n0), (k1, k0), (u1, u0)):
        assert rel_l2(a, b) <= tol


def _out(s):
    return s.cal_nlk(0.0), s.get_uk(), s.get_u(), s.get_mask()[0]


@pytest.mark.parametrize("prec", [flusi_amd.FP64, flusi_amd.FP32_MIXED])
@pytest.mark.parametrize("sponge", ["no", "cavity", "outlet_x"])
@pytest.mark.parametrize("method", ["AB2", "RK4"])
# nx = 96 with idle lanes: few lines, an odd number of waves, many; twelve
# positions a lane (2^20 points) and the other lengths, whose waves are full
@pytest.mark.parametrize("shape", [(96, 16, 16), (96, 24, 48), (96, 96, 96), (96, 96, 128), (48, 32, 32), (64, 32, 32)])
def test_sums_match_block_x_pass(tmp_path, monkeypatch, shape, method, sponge, prec):
    ini = _sphere(tmp_path, "case.ini", shape, method, sponge)
    print(f"[sums] {shape} {method} {sponge} {prec}", flush=True)
    out = []
    for wave in ("0", "1"):
        monkeypatch.setenv("FLUSI_XWAVE", wave)
        with flusi_amd.Flusi(ini, prec) as s:
            s.init_fields()
            if wave == "1":
                _fill_lds(tmp_path)
            first = s.cal_nlk(0.0)
            s.advance(STEPS)
            out.append((first,) + _out(s))
    (f0, *s0), (f1, *s1) = out
    assert np.all(np.isfinite(f1)) and rel_l2(f1, f0) <= TOL[prec]
    _check(s1, s0, prec, STEPS * STAGES[method] + 1)


@pytest.mark.parametrize("prec", [flusi_amd.FP64, flusi_amd.FP32_MIXED])
@pytest.mark.parametrize("method", ["RK2", "RK4"])
@pytest.mark.parametrize("mode", [flusi_amd.ENSEMBLE_BATCHED, flusi_amd.ENSEMBLE_GRAPH])
def test_sums_of_two_members(tmp_path, monkeypatch, mode, method, prec):
    shape = (96, 32, 48)
    inis = [_sphere(tmp_path, f"m{i}.ini", shape, method, "no", x0=0.35 + 0.1 * i) for i in range(2)]
    print(f"[sums] members {mode} {method} {prec}", flush=True)
    out = []
    for wave in ("0", "1"):
        monkeypatch.setenv("FLUSI_XWAVE", wave)
        with flusi_amd.Ensemble(inis, prec) as e:
            e.init_fields()
            assert e.batches() == [(2,) + shape]
            if wave == "1":
                _fill_lds(tmp_path)
            e.advance(STEPS, mode)
            out.append([_out(e.member(i)) for i in range(2)])
    for s0, s1 in zip(*out):
        _check(s1, s0, prec, STEPS * STAGES[method] + 1)


@pytest.mark.parametrize("prec", [flusi_amd.FP64, flusi_amd.FP32_MIXED])
def test_bumblebee_at_96(tmp_path, monkeypatch, prec):
    """The tethered bumblebee with its dynamic mean flow, twenty RK4 steps."""
    steps = 20
    ini = rewrite_ini(os.path.join(GOLDEN, "insects_flow_BB_tethered_RK4", "insect_test.ini"), str(tmp_path),
                      Resolution__nx=96, Resolution__ny=96, Resolution__nz=96, Time__dt_fixed="1.0e-3", Time__Tmax="1.0e9",
                      Time__nt=1000000, Saving__itdrag=100000, Saving__tintegral="1.0e9", Saving__tsave="1.0e9")
    print(f"[sums] bumblebee {prec}", flush=True)
    out = []
    for wave in ("0", "1"):
        monkeypatch.setenv("FLUSI_XWAVE", wave)
        with flusi_amd.Flusi(ini, prec) as s:
            s.init_fields()
            s.advance(steps)
            out.append((s.get_uk(), s.get_u()))
    (k0, u0), (k1, u1) = out
    assert np.all(np.isfinite(k1)) and np.all(np.isfinite(u1))
    tol = TOL[prec] * steps * STAGES["RK4"] / 3
    assert abs(k0[0, 0, 0, 0]) > 0.0
    assert np.max(np.abs(k1[:, 0, 0, 0] - k0[:, 0, 0, 0])) <= tol * np.max(np.abs(u0))
    assert rel_l2(k1, k0) <= tol
    assert rel_l2(u1, u0) <= tol
