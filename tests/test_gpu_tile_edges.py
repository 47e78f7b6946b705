"""The pressure solve's kernels where their tiles end: the operator stencil
on grids a cell short of, at and past its 31- and 63-cell rows, its rows in j
and its k chunks, and the y-line solve at the row counts where its chunks of
8, 16 and 32 rows fill, end and overflow.

The coarsest level in one work-group against the launches it replaces.

Tolerances: an operator apply differs from the oracle's assembled rows by
rounding only (1e-13, as in the parity tests).  A line solve differs from a
banded solve of the oracle's rows by the roundings of its own precision times
the lines' conditioning."""
import numpy as np
import pytest
from scipy.linalg import solve_banded

from curvib_old_amd import cases
from curvib_old_amd.solver import from_case as gpu_case
from oracle.pyoracle import from_case as oracle_case

pytestmark = pytest.mark.gpu

CHANNEL, BOX, OPEN = (7, 7, 1, 1, 7, 7), (1, 1, 1, 1, 1, 1), (7, 7, 1, 1, 5, 4)


def rel(a, b):
    return float(np.linalg.norm(a - b) / max(np.linalg.norm(b), 1e-300))


@pytest.mark.parametrize("cells,bctype,sphere", [
    ((4, 4, 4), CHANNEL, None), ((28, 5, 9), BOX, None), ((29, 6, 10), CHANNEL, None), ((30, 7, 11), OPEN, None),
    ((31, 9, 63), CHANNEL, None), ((60, 10, 64), BOX, (0.5, 0.5, 0.5, 0.5)), ((61, 11, 66), CHANNEL, None),
    ((62, 13, 4), CHANNEL, None), ((93, 12, 12), OPEN, (0.5, 0.5, 0.5, 0.5)), ((5, 4, 194), CHANNEL, None),
    ((6, 5, 201), BOX, None)])
def test_operator_apply_at_tile_edges(cells, bctype, sphere):
    case = cases.ChannelCase(cells=cells, amp=0.08, beta=1.5, sphere=sphere, re=300.0, seed=5, bctype=bctype, inlet=7)
    u, _ = gpu_case(case, mglevels=1)
    o, _ = oracle_case(case, nlev=1)
    try:
        o.poisson_lhs(0)
        mx, my, mz = o.dims(0)[:3]
        x = np.random.default_rng(11).standard_normal((mz, my, mx))
        e = rel(u.PoissonApply(x, 0), o.matvec(0, x))
        assert e < 1e-13, (cells, e)
    finally:
        u.close()
        o.close()


def _lines(o, case):
    """The oracle operator's coefficients of x[c-e_j], x[c], x[c+e_j] on every
    interior row, by applying it to the 27 lattices of every third point (x
    and z hold a multiple of three cells, so the periodic images keep apart)."""
    mx, my, mz = case.storage
    k, j, i = np.meshgrid(np.arange(mz), np.arange(my), np.arange(mx), indexing="ij")
    T = np.zeros((3, mz, my, mx))
    for a in range(3):
        for c in range(3):
            own = ((i - 1) % 3 == a) & ((k - 1) % 3 == c)
            for b in range(3):
                x = (own & (j % 3 == b)).astype(float)
                # ghost columns hold the images of the interior ones
                x[:, :, 0], x[:, :, -1] = x[:, :, -2], x[:, :, 1]
                x[0], x[-1] = x[-2], x[1]
                y = o.matvec(0, x)
                for q in range(3):       # coefficient of row j of the point j + q - 1
                    m = own & ((j + q - 1) % 3 == b)
                    T[q][m] = y[m]
    return T


@pytest.mark.parametrize("rows", [4, 7, 8, 9, 16, 17, 127, 128, 129, 160, 255, 256, 257, 400, 511, 513])
def test_line_solve_at_chunk_edges(rows):
    """One FGMRES iteration preconditioned by one undamped line sweep on one
    level returns a multiple of T^-1 b less its mean, T the j-tridiagonal part
    of the oracle's rows."""
    case = cases.ChannelCase(cells=(12, rows, 9), amp=0.05, beta=1.0, sphere=None, re=300.0, seed=6, dt=2e-4)
    o, _ = oracle_case(case, nlev=1)
    o.poisson_lhs(0)
    T = _lines(o, case)[:, 1:-1, 1:-1, 1:-1]
    o.close()
    for prec, eps in (("fp64", 2.0 ** -53), ("mixed", 2.0 ** -24), ("mixed16", 2.0 ** -11)):
        u, _ = gpu_case(case, mglevels=1)
        u.set_solver(precision=prec, smoother="yline", omega=1.0, coarse_sweeps=1, max_it=1, rtol=1e-30)
        u.PoissonSolver_MG(allow_unconverged=True)
        phi = u.get("phi")[1:-1, 1:-1, 1:-1]
        b = u.get("b")[1:-1, 1:-1, 1:-1]
        u.close()
        z = np.empty_like(b)
        cond = 0.0
        for k in range(b.shape[0]):
            for i in range(b.shape[2]):
                lo, dg, up = T[:, k, :, i]
                ab = np.zeros((3, rows))
                ab[0, 1:], ab[1], ab[2, :-1] = up[:-1], dg, lo[1:]
                w = solve_banded((1, 1), ab, np.stack([b[k, :, i], np.ones(rows)], axis=1))
                z[k, :, i] = w[:, 0]
                cond = max(cond, np.abs(w[:, 1]).max() * np.abs([lo, dg, up]).sum(0).max())
        z -= z.mean()
        scale = float((phi * z).sum() / (z * z).sum())
        e = rel(phi, scale * z)
        # the coefficients, the factors and the two recurrences each round once:
        # three roundings a row, amplified by the lines' conditioning
        print(f"rows {rows} {prec}: {e:.2e}, conditioning {cond:.1f}", flush=True)
        assert e < 3 * eps * cond, (rows, prec, e, cond)


@pytest.mark.parametrize("cells,bctype,sphere", [
    ((3, 4, 3), CHANNEL, None), ((8, 8, 8), BOX, (0.5, 0.5, 0.5, 0.5)), ((4, 32, 4), CHANNEL, None),
    ((5, 33, 7), OPEN, None), ((12, 8, 20), CHANNEL, (0.5, 0.5, 0.5, 0.5)), ((3, 128, 3), CHANNEL, None),
    ((3, 129, 4), BOX, None), ((3, 200, 3), CHANNEL, None), ((16, 5, 16), CHANNEL, None), ((31, 4, 14), OPEN, None)])
def test_coarsest_level_in_one_work_group_keeps_the_bits(cells, bctype, sphere):
    """The coarsest level's sweeps and nullspace rule as one work-group against
    the same as launches, which run where a kernel of that level is timed: the
    same phi bit for bit, up to the sizes where a thread takes seven faces."""
    case = cases.ChannelCase(cells=cells, amp=0.05, beta=1.0, sphere=sphere, re=300.0, seed=8, dt=2e-4, bctype=bctype,
                             inlet=7)
    u, _ = gpu_case(case, mglevels=1)
    try:
        for prec in ("fp64", "mixed", "mixed16"):
            for smoother, omega in (("yline", 0.9), ("jacobi", 0.8)):
                u.set_solver(precision=prec, smoother=smoother, omega=omega, coarse_sweeps=7, rtol=1e-8, max_it=8)
                u.prof_select("none")
                a = u.PoissonSolver_MG(allow_unconverged=True)
                phi = u.get("phi")
                u.prof_select("resid", level=0)
                b = u.PoissonSolver_MG(allow_unconverged=True)
                n = u.prof_read()[0]
                assert n >= 6, (cells, prec, smoother, n)       # the launches did run
                assert a["ksp_its"] == b["ksp_its"] and a["ksp_rnorm"] == b["ksp_rnorm"], (cells, prec, smoother, a, b)
                assert np.isfinite(phi).all() and np.array_equal(phi, u.get("phi")), (cells, prec, smoother)
    finally:
        u.close()
