"""The physical-column Crank-Nicolson solve (k_cn_phys) at the row counts where its
chunks change shape, one LES step against the oracle: fewer rows than one chunk of
9, all chunks full or all but one short, 32 and 16 columns per block, 17-row chunks,
8 columns per block; x lines of 16 points; the float increments.

Bars: u1, u2, u3, theta, nu_t 1e-11 (relative L2) in FP64; mixed 1e-6 (the float
transforms, 6e-8, times the few products they enter).  The pressure in the measure
in which it acts on the velocity, h |k dcp| / |u| with h the longest substep and k
the first mode of x, at the velocity's bar (its own relative error holds the
round-off of |u| / h_bar)."""
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


# rows = ny + 2
@pytest.mark.parametrize("nx,ny,precision", [
    (32, 6, FP64), (32, 17, FP64), (16, 17, MIXED), (16, 62, FP64), (32, 70, FP64), (32, 71, MIXED), (32, 142, FP64),
    (32, 143, FP64), (32, 143, MIXED), (32, 270, MIXED), (32, 286, FP64), (32, 287, FP64), (16, 545, FP64)])
def test_one_les_step(nx, ny, precision):
    print(f"one LES step {nx}x{ny}x16, precision {precision}", flush=True)
    c = configs.small_dns(nx, ny, 16, precision)
    c.use_les, c.les_model_type = True, 5
    p = Problem(c)
    s = p.initial_state(seed=4, theta_noise=1e-3)
    rng = np.random.default_rng(4)
    for a in (s.cu1, s.cu2, s.cu3, s.cth[0]):  # resolved modes: the model is active on most points
        shp = (ny - 3, 4, 4)
        a[2:ny - 1, 1:5, 1:5] += 0.05 * (rng.standard_normal(shp) + 1j * rng.standard_normal(shp))
    g, o = Solver(p), oracle.Oracle(Problem(c.copy(precision=FP64)), threads=16)
    o.upload_state(s)
    o.rem_div()
    s = o.download_state()
    g.upload_state(s)
    g.step(time=0.0, time_step=1, create_new_flow=False)
    for rk in (1, 2, 3):
        o.rk_substep(rk, time=0.0, time_step=1, create_new_flow=0)
    sg, so = g.download_state(), o.download_state()
    errs = {k: rel(getattr(sg, k), getattr(so, k)) for k in ("cu1", "cu2", "cu3")}
    errs["cth0"] = rel(sg.cth[0], so.cth[0])
    h = c.delta_t * 8.0 / 15.0
    speed = np.sqrt(sum(np.linalg.norm(getattr(so, k)) ** 2 for k in ("cu1", "cu2", "cu3")))
    errs["h k cp / u"] = h * p.kx[1] * np.linalg.norm(sg.cp - so.cp) / speed
    errs["nu_t"] = rel(g.download_les()[0], o.download_les()[0])
    print({k: f"{v:.1e}" for k, v in errs.items()}, flush=True)
    for k, e in errs.items():
        assert e <= (1e-11 if precision == FP64 else 1e-6), (k, e)
