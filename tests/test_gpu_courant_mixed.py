"""variable_dt on a mixed handle: the substep in which courant runs takes its own
kernels (DNS: the float column pass without its projection, then k_project; LES: the
FP64 transforms and the FP64 solve with a float eddy viscosity), against the FP64 oracle,
at row counts that take different shapes of those kernels.

Bars: delta_t is a minimum of quotients dx / |u| over points, |u| with the float
transforms' error; u1, u2, u3, theta 1e-6 (relative L2: the float transforms, 6e-8, times
the few products they enter, at steps of CFL 1/2), hence delta_t 1e-5 (a point's error
against the mean's), nu_t 1e-5."""
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


# DNS rows (ny + 2): 32 chunks, 64, tables in global memory; LES rows: 32 columns by 9
# rows, 16 by 9, 16 by 17
@pytest.mark.parametrize("les,ny", [(False, 33), (False, 161), (False, 321), (True, 33), (True, 145), (True, 290)])
def test_mixed_courant_matches_oracle(les, ny):
    print(f"mixed courant, {'LES' if les else 'DNS'} 32x{ny}x32", flush=True)
    if les:
        cfg = configs.front_les(32, ny, 32, 5000.0, 2e-4, 1e-2, precision=MIXED)
    else:
        cfg = configs.small_dns(32, ny, 32, MIXED)
    p = Problem(cfg)
    o = oracle.Oracle(Problem(cfg.copy(precision=FP64)), threads=16)
    s = p.initial_state(seed=5, theta_noise=1e-3)
    rng = np.random.default_rng(5)
    sh = (ny - 3, 3, 3)
    for a in (s.cu1, s.cu2, s.cu3):
        a[2:ny - 1, 1:4, 1:4] += 0.3 * (rng.standard_normal(sh) + 1j * rng.standard_normal(sh))
    o.upload_state(s)
    o.rem_div()
    s = o.download_state()
    g = Solver(p)
    g.upload_state(s)
    g.set_variable_dt(True, 1, 0.5)
    o.set_variable_dt(True, 1, 0.5)
    t, dt = 0.0, cfg.delta_t
    for n in (1, 2):
        for rk in (1, 2, 3):
            g.rk_substep(rk, delta_t=dt, time=t, time_step=n, create_new_flow=not les)
            o.rk_substep(rk, delta_t=dt, time=t, time_step=n, create_new_flow=int(not les))
        (dg, rg), (do, ro) = g.courant(t, 10.0, 100.0, 100.0), o.courant(t, 10.0, 100.0, 100.0)
        print(f"step {n}: dt {dg!r} {do!r}", flush=True)
        assert rg and ro and do > 0 and abs(dg - do) <= 1e-5 * do
        t += dt
        dt = do
    sg, so = g.download_state(), o.download_state()
    errs = {k: rel(getattr(sg, k), getattr(so, k)) for k in ("cu1", "cu2", "cu3")}
    errs["cth0"] = rel(sg.cth[0], so.cth[0])
    print({k: f"{v:.1e}" for k, v in errs.items()}, flush=True)
    for k, e in errs.items():
        assert e <= 1e-6, (k, e)
    if les:
        nu = o.download_les()[0]
        assert (nu > 0).mean() > 0.1 and rel(g.download_les()[0], nu) <= 1e-5
