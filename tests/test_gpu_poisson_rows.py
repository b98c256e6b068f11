"""dgpu_poisson_p at the row and scalar counts where k_project's chunks change shape
(chunks without rows, one, two, three and five rows each, 64 chunks, tables in global
memory), against the oracle.

Bar: 1e-11, relative max on rows 1..Nyp, as at 32x33x32 (the solve of projection tests
at up to 385 rows)."""
import numpy as np
import pytest

import oracle
from diablo3_amd import configs
from diablo3_amd.problem import Problem
from diablo3_amd.solver import Solver
from oracle import flow_io as ofi

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("ny,n_th", [(4, 1), (17, 2), (30, 0), (31, 1), (65, 2), (158, 1), (159, 2), (319, 1)])
def test_poisson_p(ny, n_th):
    print(f"poisson_p 16x{ny}x16, {n_th} scalars", flush=True)
    n = n_th
    c = configs.small_dns(16, ny, 16)
    c = c.copy(n_th=n, ri=[1.0] * n, pr=[1.0, 0.7][:n], create_new_th=[True] * n, th_bc_ymin=[1, 0][:n],
               th_bc_ymin_c1=[1.0, 0.3][:n], th_bc_ymax=[1, 0][:n], th_bc_ymax_c1=[1.0, 0.2][:n],
               dthdx=[0.5, 0.1][:n], dthdz=[0.0, 0.2][:n]).derive()
    p = Problem(c)
    s = p.initial_state(seed=4, theta_noise=1e-2)
    rng = np.random.default_rng(4)
    for a in (s.cu1, s.cu2, s.cu3, *s.cth):
        shp = (max(ny - 3, 1), 3, 3)
        a[2:max(ny - 1, 3), 1:4, 1:4] += 0.1 * (rng.standard_normal(shp) + 1j * rng.standard_normal(shp))
    g, o = Solver(p), oracle.Oracle(p, threads=16)
    g.upload_state(s)
    g.rem_div()
    s = g.download_state()
    o.upload_state(s)
    want = ofi.poisson_p(o)[1:ny + 1]
    g.poisson_p()
    r = g.download_state()
    err = np.abs(r.cp[1:ny + 1] - want).max() / np.abs(want).max()
    print(f"cp {err:.2e}", flush=True)
    assert err <= 1e-11
    for a, b in ((r.cu1, s.cu1), (r.cu2, s.cu2), (r.cu3, s.cu3), *zip(r.cth, s.cth)):
        assert np.array_equal(a, b)
