"""A step at nz = 1024, where the z transforms have threads, tiles and persistence of
their own in each precision, against the oracle (DNS and LES).

Bars (relative L2): FP64 1e-11, as for a step at any size; mixed DNS 1e-8 (the float
transforms enter u through dt NL, 6e-8 x dt x |NL| / |u|), mixed LES 1e-6 (the whole
increment goes through them); nu_t 1e-11 and 1e-5."""
import numpy as np
import pytest

import oracle
from diablo3_amd import configs
from diablo3_amd.config import FP64, MIXED
from diablo3_amd.problem import Problem
from diablo3_amd.solver import Solver

pytestmark = pytest.mark.gpu


def rel(a, b):
    return np.linalg.norm(a - b) / max(np.linalg.norm(b), 1e-300)


@pytest.mark.parametrize("les,precision", [(False, FP64), (False, MIXED), (True, FP64), (True, MIXED)])
def test_one_step(les, precision):
    nx, ny, nz = 16, 9, 1024
    print(f"one {'LES' if les else 'DNS'} step {nx}x{ny}x{nz}, precision {precision}", flush=True)
    c = configs.small_dns(nx, ny, nz, precision)
    c.use_les, c.les_model_type = les, 5
    p = Problem(c)
    s = p.initial_state(seed=6, theta_noise=1e-3)
    rng = np.random.default_rng(6)
    for a in (s.cu1, s.cu2, s.cu3, s.cth[0]):  # every kept kz, so that a misplaced row shows
        shp = (6, c.kzr, 4)
        a[2:8, :, 1:5] += 2e-3 * (rng.standard_normal(shp) + 1j * rng.standard_normal(shp))
    g, o = Solver(p), oracle.Oracle(Problem(c.copy(precision=FP64)), threads=16)
    o.upload_state(s)
    o.rem_div()
    s = o.download_state()
    g.upload_state(s)
    g.step(time=0.0, time_step=1, create_new_flow=not les)
    for rk in (1, 2, 3):
        o.rk_substep(rk, time=0.0, time_step=1, create_new_flow=int(not les))
    sg, so = g.download_state(), o.download_state()
    errs = {k: rel(getattr(sg, k), getattr(so, k)) for k in ("cu1", "cu2", "cu3")}
    errs["cth0"] = rel(sg.cth[0], so.cth[0])
    nu = rel(g.download_les()[0], o.download_les()[0]) if les else 0.0
    print({k: f"{v:.1e}" for k, v in errs.items()}, f"nu_t {nu:.1e}", flush=True)
    bar = 1e-11 if precision == FP64 else (1e-6 if les else 1e-8)
    for k, e in errs.items():
        assert e <= bar, (k, e)
    assert nu <= (1e-11 if precision == FP64 else 1e-5)
