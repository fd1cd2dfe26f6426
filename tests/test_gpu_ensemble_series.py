"""The time series of ensemble members: batched and graph-replayed steps write
every member's ekin.t as its own steps do."""
import os

import numpy as np
import pytest

import flusi_amd
from flusi_amd.ensemble_configs import write_ensemble

pytestmark = pytest.mark.gpu

MODES = (flusi_amd.ENSEMBLE_MEMBERS, flusi_amd.ENSEMBLE_BATCHED, flusi_amd.ENSEMBLE_GRAPH)


@pytest.mark.parametrize("prec", [flusi_amd.FP64, flusi_amd.FP32_MIXED])
@pytest.mark.parametrize("method", ["RK2", "RK4"])
@pytest.mark.parametrize("between", ["nothing", "rhs", "set_uk"])
def test_ekin_of_members(tmp_path, between, method, prec):
    """Also after a right-hand side (whose z step writes no energies) and after
    a state was set (whose first step sums the energies of other tiles)."""
    paths = write_ensemble(str(tmp_path / "ini"), sizes=(32, 64), per_size=4, dt=5.0e-4, nt=50, method=method)
    print(f"[series] {between} {method} {prec}", flush=True)
    files = []
    for mode in MODES:
        dirs = [str(tmp_path / f"{mode}_{i}") for i in range(len(paths))]
        with flusi_amd.Ensemble(paths, prec) as e:
            for i, d in enumerate(dirs):
                os.makedirs(d)
                e.member(i).set_output_dir(d)
            e.init_fields()
            e.advance(3, mode)
            for i in range(e.n):
                m = e.member(i)
                if between == "rhs":
                    m.cal_nlk(m.get_time()[0])
                elif between == "set_uk":
                    m.set_uk(m.get_uk())
            e.advance(3, mode)
            last = [e.member(i).energy_k() for i in range(e.n)]
        rows = [np.loadtxt(os.path.join(d, "ekin.t"), comments="%") for d in dirs]
        for r, k in zip(rows, last):
            assert r.shape == (6, 2)
            # eight digits in the file
            assert abs(r[-1, 1] - k) <= 2e-8 * k
        files.append([open(os.path.join(d, "ekin.t")).read() for d in dirs])
    assert files[1] == files[0]
    assert files[2] == files[0]
