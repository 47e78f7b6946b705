"""A context that changes its solver's precision solves with the operator of the
precision it has now: the FP16 coefficients and line factors that CV_MIXED16
left behind are neither used nor kept across a new body.  Tolerance: exact
equality with a context that never had another precision."""
import numpy as np
import pytest

from curvib_old_amd import cases
from curvib_old_amd.solver import from_case

pytestmark = pytest.mark.gpu

OPTS = dict(smoother="yline", omega=0.9, pre_sweeps=3, post_sweeps=3, coarse_sweeps=10, rtol=1e-8, max_it=6)


# 24 rows on small levels (one-launch sweeps, coarsest level in one work-group), 140 and 300 rows (16 and 32 a
# thread), a finest level of more than 400,000 points (line solves as launches)
@pytest.mark.parametrize("cells", [(16, 24, 16), (12, 140, 8), (6, 300, 8), (62, 102, 62)])
@pytest.mark.parametrize("before,now", [("mixed16", "mixed"), ("mixed16", "fp64"), ("mixed", "mixed16")])
def test_solves_follow_the_current_precision(cells, before, now):
    case = cases.ChannelCase(cells=cells, amp=0.05, sphere=(0.5, 0.5, 0.5, 0.5), re=300.0, seed=8, dt=2e-4)
    (u, (_, nv, _)), (fresh, _) = (from_case(case, mglevels=2, semi=(1, 1, 0)) for _ in range(2))
    try:
        u.set_solver(precision=before, **OPTS)
        u.PoissonSolver_MG(allow_unconverged=True)
        u.set_solver(precision=now, **OPTS)
        fresh.set_solver(precision=now, **OPTS)
        for body in (nv, np.where(nv > 0.1, 0.0, nv)):
            for c in (u, fresh):
                c.set_nvert(body)
            a, b = (c.PoissonSolver_MG(allow_unconverged=True) for c in (u, fresh))
            assert a["ksp_its"] == b["ksp_its"] and a["ksp_rnorm"] == b["ksp_rnorm"], (cells, before, now, a, b)
            phi = fresh.get("phi")
            assert np.isfinite(phi).all() and np.array_equal(u.get("phi"), phi), (cells, before, now)
    finally:
        u.close()
        fresh.close()
