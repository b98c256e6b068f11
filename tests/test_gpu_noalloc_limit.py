"""The size limit of dgpu_fft_xz_to_fourier_noalloc at its edge: field, x-spectra and
spectrum (each rounded up to 256 bytes) of 128 x Ny x 128 fit 64 MiB up to 227 rows and
not at 228; the refusal names the limit, and does not call those bytes a need."""
import numpy as np
import pytest

from diablo3_amd import configs, layout
from diablo3_amd.problem import Problem
from diablo3_amd.solver import Solver, load
from test_zz_no_alloc import DevBuf, _hip, _noalloc

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("ny,accepted", [(225, True), (226, False)])
def test_limit(ny, accepted):
    cfg = configs.small_dns(128, ny, 128)
    sizes = [8 * 128 * 128 * cfg.ny2, 16 * 48 * 128 * cfg.ny2, 16 * 48 * cfg.kzr * cfg.ny2]
    total = sum((b + 255) // 256 * 256 for b in sizes)
    assert (total <= 64 << 20) == accepted
    g = Solver(Problem(cfg))
    hip = _hip()
    buf = DevBuf(hip, np.zeros(layout.fortran_physical_shape(cfg)))
    rc = _noalloc(g, buf, buf)
    msg = load().dgpu_last_error().decode()
    print(ny, rc, msg, flush=True)
    buf.free()
    g.close()
    assert rc == (0 if accepted else 2)
    if not accepted:
        assert "limit" in msg and str(total) in msg and "needs" not in msg
