"""ImpRK where the tiles of its marches end: grids a cell short of, at and past
64 columns, 4 rows and a chunk of k planes, with walls, periodic pairs and an
inlet and outlet around them, so that the interior cells (CalcRHS formed in the
FormFunction1 pass) and the shell of points around them (a pass of their own)
meet on every kind of face.

Against the oracle after each converged step (both at rtol 1e-13): 1e-10
relative L2, as the other step tests.  The fused stage update against the
update and Contra2Cart as passes of their own: exact equality."""
import numpy as np
import pytest

from curvib_old_amd import cases
from curvib_old_amd.solver import from_case as gpu_case
from oracle.pyoracle import from_case as oracle_case
from conftest import assert_fields_match

pytestmark = pytest.mark.gpu

CHANNEL, BOX, OPEN = (7, 7, 1, 1, 7, 7), (1, 1, 1, 1, 1, 1), (7, 7, 1, 1, 5, 4)
IMP = dict(imp_max_it=20, imp_atol=1e-7, imp_rtol=1e-4, cfl=0.3)


def ctxs(cells, bctype, sphere, make, **kw):
    case = cases.ChannelCase(cells=cells, amp=0.08, beta=1.5, re=400.0, seed=12, dt=2e-4, bctype=bctype, inlet=7,
                             inlet_center=(0.0, 0.5, 0.0), sphere=sphere)
    u, _ = make(case, **kw)
    u.set_momentum("imprk", **IMP)
    u.set_solver(rtol=1e-13, max_it=400)
    return u


@pytest.mark.parametrize("cells,bctype,sphere", [
    ((61, 7, 14), CHANNEL, None), ((62, 6, 16), BOX, None), ((63, 5, 18), CHANNEL, None),
    ((64, 10, 8), OPEN, None), ((12, 9, 34), BOX, (0.5, 0.5, 0.5, 0.5))])
def test_imprk_at_tile_edges_tracks_the_oracle(cells, bctype, sphere):
    u = ctxs(cells, bctype, sphere, gpu_case, mglevels=1)
    o = ctxs(cells, bctype, sphere, oracle_case, nlev=1)
    try:
        for s in range(2):
            st = u.Flow_Solver()
            o.call("o_flow_step")
            so = o.imp_stats()
            assert st["imp_its"] == int(so["its"]) and st["imp_lambda"] == so["lambda"], (cells, s, st, so)
            assert_fields_match(f"imprk {cells} {bctype} step {s}", u, o)
    finally:
        u.close()
        o.close()


@pytest.mark.parametrize("cells,bctype,sphere", [
    ((61, 7, 14), CHANNEL, None), ((64, 10, 18), BOX, None), ((40, 24, 20), CHANNEL, (0.5, 0.5, 0.5, 0.5))])
def test_imprk_fused_stage_keeps_the_bits(monkeypatch, cells, bctype, sphere):
    got = []
    for fused in ("1", "0"):
        monkeypatch.setenv("CV_RK_FUSED", fused)
        u = ctxs(cells, bctype, sphere, gpu_case, mglevels=2, semi=(1, 1, 0))
        for _ in range(2):
            st = u.Flow_Solver()
        got.append((st["imp_its"], *(u.get(f) for f in ("ucont", "ucat", "p"))))
        u.close()
    assert got[0][0] == got[1][0] >= 1
    for a, b in zip(got[0][1:], got[1][1:]):
        assert np.isfinite(a).all() and np.array_equal(a, b), cells
