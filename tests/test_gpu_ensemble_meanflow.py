"""Members of a batch with a dynamic mean flow, whose zero mode takes the x
pass's penalisation sums: batched and graph-replayed steps agree with each
member's own bit for bit, so the order of those sums must not depend on the
batch."""
import os

import numpy as np
import pytest

import flusi_amd
from tests._util import CONFIGS, rewrite_ini

pytestmark = pytest.mark.gpu


# one wave a block alone and four in a batch (64^3 FP64, 96^3 FP32), one in
# both (32^3), four in both (64 x 128 x 128), the x pass of idle lanes (96)
@pytest.mark.parametrize("prec", [flusi_amd.FP64, flusi_amd.FP32_MIXED])
@pytest.mark.parametrize("shape", [(32, 32, 32), (48, 48, 48), (64, 64, 64), (96, 96, 96), (64, 128, 128)])
@pytest.mark.parametrize("members", [2, 3])
def test_members_agree_bit_for_bit(tmp_path, members, shape, prec):
    nx, ny, nz = shape
    h = 2.0 / min(ny, nz)
    inis = [rewrite_ini(os.path.join(CONFIGS, "cfg2_sphere_256x128x128.ini"), str(tmp_path), name=f"m{i}.ini",
                        Resolution__nx=nx, Resolution__ny=ny, Resolution__nz=nz, Geometry__xl=repr(nx * h),
                        Geometry__yl=repr(ny * h), Geometry__zl=repr(nz * h), Geometry__x0=repr((0.3 + 0.07 * i) * nx * h),
                        Geometry__y0=repr(0.52 * ny * h), Geometry__z0=repr(0.47 * nz * h), Geometry__Size="1.7",
                        Time__dt_fixed="5.0e-4", Sponge__iVorticitySponge="no", MeanFlow__iMeanFlow_x="dynamic",
                        MeanFlow__iMeanFlow_y="dynamic", MeanFlow__uy="0.3", MeanFlow__m_fluid="4.0",
                        Saving__tintegral=100.0, Saving__itdrag=100000) for i in range(members)]
    print(f"[meanflow] {shape} {members} {prec}", flush=True)
    out = []
    for mode in (flusi_amd.ENSEMBLE_MEMBERS, flusi_amd.ENSEMBLE_BATCHED, flusi_amd.ENSEMBLE_GRAPH):
        with flusi_amd.Ensemble(inis, prec) as e:
            e.init_fields()
            e.advance(20, mode)
            out.append([e.member(i).get_uk() for i in range(members)])
    for i in range(members):
        assert out[0][i][0, 0, 0, 0] != 1.0 and np.all(np.isfinite(out[0][i]))
        for o in out[1:]:
            assert np.array_equal(o[i], out[0][i]), float(np.max(np.abs(o[i] - out[0][i])))
