"""The LES x pass (k_les_products: model, products and their x transforms) at the line
lengths and scalar counts where its launch changes, one step against the oracle:
x lines shorter than a block, exactly one and several points per thread, the tile in
one piece and in two, 0 to 2 scalars (the second with wall conditions of its own), each
model.

Bars: u1, u2, u3, the scalars, nu_t, kappa_t 1e-11 (relative L2) in FP64, as for a step
at any size (the arithmetic per point does not depend on the size); mixed 1e-6 (the
float transforms, 6e-8, times the few products they enter), nu_t and kappa_t 1e-5."""
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


@pytest.mark.parametrize("nx,nz,n_th,model,precision", [
    (16, 16, 0, 5, FP64), (32, 32, 2, 4, FP64), (64, 16, 1, 1, MIXED), (64, 16, 2, 5, FP64), (128, 16, 1, 5, FP64),
    (256, 16, 2, 4, FP64), (512, 16, 0, 1, FP64), (512, 16, 1, 1, FP64), (512, 32, 1, 4, FP64), (512, 16, 2, 5, FP64),
    (512, 16, 2, 5, MIXED), (1024, 16, 0, 5, FP64), (1024, 16, 0, 4, MIXED), (1024, 16, 1, 5, MIXED),
    (1024, 16, 2, 1, MIXED)])
def test_one_les_step(nx, nz, n_th, model, precision):
    print(f"one LES step {nx}x9x{nz}, {n_th} scalars, model {model}, precision {precision}", flush=True)
    c = configs.small_dns(nx, 9, nz, precision)
    c.use_les, c.les_model_type = True, model
    n = n_th
    c = c.copy(n_th=n, ri=[1.0] * n, pr=[1.0, 0.7][:n], create_new_th=[True] * n, th_bc_ymin=[1, 0][:n],
               th_bc_ymin_c1=[1.0, 0.3][:n], th_bc_ymax=[1, 0][:n],
               th_bc_ymax_c1=[1.0, 0.2][:n], dthdx=[0.5, 0.1][:n],
               dthdz=[0.0, 0.2][:n]).derive()
    p = Problem(c)
    s = p.initial_state(seed=5, theta_noise=1e-3)
    rng = np.random.default_rng(5)
    for a in (s.cu1, s.cu2, s.cu3, *s.cth):  # resolved modes: the model is active on most points
        shp = (6, 4, 4)
        a[2:8, 1:5, 1:5] += 0.05 * (rng.standard_normal(shp) + 1j * rng.standard_normal(shp))
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
    errs.update({f"cth{k}": rel(sg.cth[k], so.cth[k]) for k in range(n)})
    (ntg, ktg), (nto, kto) = g.download_les(), o.download_les()
    coef = {"nu_t": rel(ntg, nto), **{f"kappa_t{k}": rel(ktg[k], kto[k]) for k in range(n)}}
    print({k: f"{v:.1e}" for k, v in {**errs, **coef}.items()}, flush=True)
    assert (nto > 0).mean() > 0.1
    for k, e in errs.items():
        assert e <= (1e-11 if precision == FP64 else 1e-6), (k, e)
    for k, e in coef.items():
        assert e <= (1e-11 if precision == FP64 else 1e-5), (k, e)
