"""A smoothing sweep of a small level as one launch (cv_sweep.h) against the
residual and line-solve launches it replaces: where its patches of 4 and 8
columns, its 64 and 128 rows and its chunks of 8 and 16 rows end, at odd and
even sweep counts, alone and in batches whose depths mix cases that take it,
cases that do not and cases that bottom out.  Tolerance: exact equality."""
import numpy as np
import pytest

from curvib_old_amd import cases
from curvib_old_amd.solver import Batch, from_case

pytestmark = pytest.mark.gpu

CHANNEL, BOX, OPEN = (7, 7, 1, 1, 7, 7), (1, 1, 1, 1, 1, 1), (7, 7, 1, 1, 5, 4)
BODY = (0.5, 0.5, 0.5, 0.5)


def case_of(cells, bctype=CHANNEL, sphere=None):
    return cases.ChannelCase(cells=cells, amp=0.05, beta=1.0, sphere=sphere, re=300.0, seed=8, dt=2e-4, bctype=bctype,
                             inlet=7)


# z alone is coarsened (even, x any size); 61 x 102 x 62 cells hold 419,328
# points: past the limit, launches on both sides
@pytest.mark.parametrize("cells,bctype,sphere", [
    ((4, 3, 6), CHANNEL, None), ((6, 8, 6), BOX, None), ((7, 9, 8), OPEN, None), ((14, 63, 6), CHANNEL, None),
    ((16, 64, 10), BOX, BODY), ((15, 65, 8), CHANNEL, None), ((10, 66, 16), OPEN, BODY), ((6, 128, 10), CHANNEL, BODY),
    ((9, 129, 6), BOX, None), ((4, 255, 6), CHANNEL, None), ((5, 256, 6), CHANNEL, None), ((4, 257, 6), CHANNEL, None),
    ((61, 102, 62), CHANNEL, BODY), ((60, 100, 60), OPEN, BODY)])
def test_sweep_in_one_launch_keeps_the_bits(cells, bctype, sphere):
    u, _ = from_case(case_of(cells, bctype, sphere), mglevels=2, semi=(1, 1, 0))
    try:
        for prec in ("fp64", "mixed", "mixed16"):
            for pre, post in ((3, 3), (2, 1)):
                u.set_solver(precision=prec, smoother="yline", omega=0.9, pre_sweeps=pre, post_sweeps=post,
                             coarse_sweeps=5, rtol=1e-8, max_it=6)
                u.prof_select("none")
                a = u.PoissonSolver_MG(allow_unconverged=True)
                phi = u.get("phi")
                u.prof_select("line", level=1)     # a timed kernel stays a launch of its own
                b = u.PoissonSolver_MG(allow_unconverged=True)
                n = u.prof_read()[0]
                assert n >= (pre + post) * a["ksp_its"], (cells, prec, n)
                assert a["ksp_its"] == b["ksp_its"] and a["ksp_rnorm"] == b["ksp_rnorm"], (cells, prec, a, b)
                assert np.isfinite(phi).all() and np.array_equal(phi, u.get("phi")), (cells, prec, pre, post)
    finally:
        u.close()


# cells and levels: depths past the limit together, a case bottoming out beside
# deeper ones, short and tall lines in one launch
GROUPS = {
    "small": [((16, 24, 16), 3), ((24, 40, 16), 3), ((16, 70, 24), 2)],
    "mixed": [((96, 66, 64), 4), ((48, 40, 48), 1), ((32, 140, 32), 3)],
    "tail": [((96, 66, 64), 3), ((24, 48, 24), 1), ((32, 24, 32), 2)],
}


@pytest.mark.parametrize("group,precision,pre,post,coarse", [
    ("small", "mixed16", 3, 3, 10), ("small", "fp64", 2, 1, 3), ("mixed", "mixed16", 3, 3, 10),
    ("mixed", "mixed", 1, 2, 4), ("tail", "mixed16", 3, 3, 10), ("tail", "fp64", 2, 3, 7)])
def test_batched_sweeps_match_each_case_alone(group, precision, pre, post, coarse):
    def ctx(cells, levels):
        u, _ = from_case(case_of(cells), mglevels=levels, semi=(0, 1, 0))
        u.set_solver(precision=precision, smoother="yline", omega=0.9, pre_sweeps=pre, post_sweeps=post,
                     coarse_sweeps=coarse, rtol=1e-7, max_it=60)
        return u

    inb, alone = ([ctx(*g) for g in GROUPS[group]] for _ in range(2))
    b = Batch(inb)
    try:
        for s in range(2):
            sb = b.step()
            for q, u in enumerate(alone):
                sa = u.Flow_Solver()
                assert sb[q]["ksp_its"] == sa["ksp_its"] and sb[q]["ksp_rnorm"] == sa["ksp_rnorm"], (s, q)
            for q, (ua, ub) in enumerate(zip(inb, alone)):
                for f in ("phi", "p", "ucont"):
                    assert np.array_equal(ua.get(f), ub.get(f)), (group, s, q, f)
    finally:
        b.close()
        for u in inb + alone:
            u.close()
