"""dgpu_timing_read's names on the paths of a step: every name is a kernel of the
sources (or one of the two groups of launches, les_grad and les_cn_fft), and bench.py's
byte model has it; a DNS substep in which courant runs times the column pass and the
projection after it."""
import os
import re

import numpy as np
import pytest

import bench
from diablo3_amd import configs
from diablo3_amd.config import MIXED
from diablo3_amd.problem import Problem
from diablo3_amd.solver import Solver

pytestmark = pytest.mark.gpu

CSRC = os.path.join(os.path.dirname(os.path.dirname(os.path.abspath(__file__))), "diablo3_amd", "csrc")


def kernels():
    src = "".join(open(os.path.join(CSRC, f)).read() for f in sorted(os.listdir(CSRC)) if f.endswith((".hip", ".hpp")))
    return set(re.findall(r"__global__[^;{]*?\bvoid\s+(k_\w+)\s*\(", src))


@pytest.mark.parametrize("les,courant", [(False, False), (False, True), (True, False)])
def test_names(les, courant):
    cfg = configs.front_les(32, 17, 32, 5000.0, 2e-4, 1e-2, precision=MIXED) if les else configs.small_dns(32, 17, 32)
    p = Problem(cfg)
    g = Solver(p)
    g.upload_state(p.initial_state(seed=2))
    g.rem_div()
    if courant:
        g.set_variable_dt(True, 1, 0.5)
    g.timing(True)
    g.step(time=0.0, time_step=1, create_new_flow=not les)
    t = g.timing_read()
    print(sorted(t), flush=True)
    assert set(t) - {"les_grad", "les_cn_fft"} <= kernels()
    assert set(t) <= set(bench.kernel_bytes(cfg, cfg.precision == MIXED))
    assert all(np.isfinite(ms) and ms > 0 for ms, _ in t.values())
    if not les:
        assert t["k_column"][1] == 3
        assert ("k_project" in t) == courant
