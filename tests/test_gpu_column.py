"""The column kernels (k_column, k_project) at the row counts where their chunks
change shape, against the oracle through the C ABI: fewer rows than chunks, chunks
all full or all but one short, the steps from 32 to 64 chunks and from tables in
LDS to tables in global memory (4 and 2 columns per block).

Bars: u1, u2, u3, theta 1e-11 (relative L2) after the projection and after one
FP64 step; mixed 1e-8 (the float transforms enter u through dt NL, 6e-8 x dt x
|NL| / |u|).  The pressure is phi / h_bar of a flow that starts without one, so its
relative error holds the round-off of |u| / h_bar over a small |cp| (up to 2e-9
here, the same with Thomas sweeps on either side); it acts on the velocity as
h_bar grad cp, and in that measure it is held to the velocity's bar: h |k cp error|
against |u|, h the longest substep and k the first mode of x (y gradients of the
error vanish with it: phi is smooth between walls)."""
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


def problem(ny, n_th, precision):
    c = configs.small_dns(16, ny, 16, precision)
    n = n_th
    c = c.copy(n_th=n, ri=[1.0] * n, pr=[1.0, 0.7][:n], create_new_th=[True] * n, th_bc_ymin=[1, 0][:n],
               th_bc_ymin_c1=[1.0, 0.3][:n], th_bc_ymax=[1, 0][:n], th_bc_ymax_c1=[1.0, 0.2][:n],
               dthdx=[0.5, 0.1][:n], dthdz=[0.0, 0.2][:n]).derive()
    return Problem(c)


# rows = ny + 2: 6 and 19 (chunks without rows), 32 (one row each), 33, 64 (two each),
# 159, 160, 161 (64 chunks), 320, 321 (global tables, 4 columns), 643 (2 columns)
@pytest.mark.parametrize("ny,n_th,precision", [
    (4, 1, FP64), (17, 2, FP64), (30, 1, FP64), (31, 0, FP64), (62, 1, MIXED), (157, 2, FP64), (158, 1, FP64),
    (159, 1, FP64), (159, 2, MIXED), (318, 1, FP64), (319, 1, FP64), (319, 2, MIXED), (641, 1, FP64)])
def test_one_step(ny, n_th, precision):
    print(f"one step 16x{ny}x16, {n_th} scalars, precision {precision}", flush=True)
    p = problem(ny, n_th, precision)
    g, o = Solver(p), oracle.Oracle(Problem(p.cfg.copy(precision=FP64)), threads=16)
    s = p.initial_state(seed=3, theta_noise=1e-3)
    o.upload_state(s)
    o.rem_div()
    g.upload_state(s)
    g.rem_div()
    sg, so = g.download_state(), o.download_state()
    for k in ("cu1", "cu2", "cu3"):
        assert rel(getattr(sg, k), getattr(so, k)) <= 1e-11, ("projection", k)
    g.upload_state(so)
    g.step(time=0.0, time_step=1)
    o.step(time=0.0, time_step=1)
    sg, so = g.download_state(), o.download_state()
    errs = {k: rel(getattr(sg, k), getattr(so, k)) for k in ("cu1", "cu2", "cu3")}
    h = p.cfg.delta_t * 8.0 / 15.0
    speed = np.sqrt(sum(np.linalg.norm(getattr(so, k)) ** 2 for k in ("cu1", "cu2", "cu3")))
    errs["h k cp / u"] = h * p.kx[1] * np.linalg.norm(sg.cp - so.cp) / speed
    errs.update({f"cth{n}": rel(sg.cth[n], so.cth[n]) for n in range(n_th)})
    print({k: f"{v:.1e}" for k, v in errs.items()}, flush=True)
    for k, e in errs.items():
        assert e <= (1e-11 if precision == FP64 else 1e-8), (k, e)
