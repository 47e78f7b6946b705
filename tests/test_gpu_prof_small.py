"""Timing the kernels that small levels run: the one-launch sweeps and the coarsest
level in one work-group are timed as such, and neither that nor timing a kernel
they do not hold changes what runs.  The counts follow from the cycle: per FGMRES
iteration one V-cycle, whose first pre-sweep starts from zero and is a line solve
alone.  The face RHS counts the values CalcRHS reads beside its own: in ImpRK Ucont of
this and the last step, from the second step on of the one before too.  Tolerance:
exact equality."""
import numpy as np
import pytest

from curvib_old_amd import cases
from curvib_old_amd.solver import from_case

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("precision", ["fp64", "mixed", "mixed16"])
# the coarsest level holds 4 x 24 x 8 and 8 x 24 x 8 cells, 2600 and 5056 faces (7168 fit)
@pytest.mark.parametrize("cells,levels", [((16, 24, 8), 3), ((8, 24, 8), 1)])
def test_small_levels_kernels_are_timed(precision, cells, levels):
    case = cases.ChannelCase(cells=cells, amp=0.05, re=300.0, seed=8, dt=2e-4)
    u, _ = from_case(case, mglevels=levels, semi=(0, 1, 1))
    try:
        u.set_solver(precision=precision, smoother="yline", omega=0.9, pre_sweeps=3, post_sweeps=2, coarse_sweeps=5,
                     rtol=1e-7, max_it=8)

        def solve(kernel, level=-1):
            u.prof_select(kernel, level=level)
            st = u.PoissonSolver_MG(allow_unconverged=True)
            n, ms, nbytes = u.prof_read()
            assert (n > 0) == (ms > 0) == (nbytes > 0), (kernel, n, ms, nbytes)
            return st["ksp_its"], st["ksp_rnorm"], u.get("phi"), n

        its, rnorm, phi, _ = solve("none")
        top = levels - 1
        want = {("coarse", 0): its, ("coarse", top): its if levels == 1 else 0,
                ("sweep", top): 0 if levels == 1 else (3 + 2 - 1) * its, ("line", top): None, ("resid", 0): None,
                ("orth", -1): None, ("apply", -1): its}   # orth: a second pass where the first cancels
        for (kernel, level), n in want.items():
            i, r, p, got = solve(kernel, level)
            assert i == its and r == rnorm and np.array_equal(p, phi), (precision, kernel, level)
            assert got == n if n is not None else got > 0, (precision, kernel, level, got, n)
    finally:
        u.close()


def test_face_rhs_counts_calcrhs_bytes():
    case = cases.ChannelCase(cells=(16, 24, 8), amp=0.05, re=300.0, seed=8, dt=2e-4)
    u, _ = from_case(case, mglevels=1)
    try:
        u.set_solver(smoother="yline", rtol=1e-6)
        u.prof_select("ff1")
        u.Flow_Solver()
        n, _, nbytes = u.prof_read(reset=True)
        pts = np.prod(case.storage)
        assert n == 4 and nbytes == n * pts * (17 * 8 + 4)
        u.put("ucont", u.get("ucont"))      # a first step again
        u.set_momentum(scheme="imprk")
        for values in (17 + 6, 17 + 9):
            u.Flow_Solver()
            n, _, nbytes = u.prof_read(reset=True)
            assert n > 4 and nbytes == n * pts * (values * 8 + 4), (n, nbytes / n / pts, values)
    finally:
        u.close()
