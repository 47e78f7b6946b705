"""cv_divergence_noalloc where its tiles end: storage extents at, below and past
the 64 columns, 4 or 16 rows and 16 planes of a tile, the grids that take the
small and the large tiles, ties, an all-zero field and a NaN, against the same
expression in numpy.

The value is one rounding away from numpy's at most where the compiler fuses
the last product (the sum of six fluxes times 1/J: relative 2^-50 of the largest
term); the index is exact, the inputs keeping the largest value apart."""
import ctypes as C

import numpy as np
import pytest

from curvib_old_amd import _lib

pytestmark = pytest.mark.gpu
torch = pytest.importorskip("torch")


def device(u, aj, nv):
    t = [torch.as_tensor(a, device="cuda").contiguous() for a in (u, aj, nv)]
    out = torch.full((2,), -7.0, dtype=torch.float64, device="cuda")
    mz, my, mx = aj.shape
    rc = _lib.load().cv_divergence_noalloc(0, *(C.c_void_p(a.data_ptr()) for a in t), mx, my, mz,
                                           C.c_void_p(torch.cuda.current_stream().cuda_stream),
                                           C.c_void_p(out.data_ptr()))
    assert rc == _lib.CV_OK, _lib.last_error()
    v, i = out.tolist()
    return v, int(i)


def host(u, aj, nv):
    c, lo, hi = slice(1, -1), slice(0, -2), slice(2, None)
    d = np.zeros_like(aj)
    d[c, c, c] = np.abs((u[c, c, c, 0] - u[c, c, lo, 0] + u[c, c, c, 1] - u[c, lo, c, 1] + u[c, c, c, 2] -
                         u[lo, c, c, 2]) * aj[c, c, c])
    near = nv[c, c, c] + nv[hi, c, c] + nv[lo, c, c] + nv[c, hi, c] + nv[c, lo, c] + nv[c, c, hi] + nv[c, c, lo]
    d[c, c, c][near > 0.1] = 0.0
    i = int(d.argmax())
    return float(d.reshape(-1)[i]), i


@pytest.mark.parametrize("storage", [(3, 3, 3), (5, 4, 3), (65, 6, 17), (66, 7, 18), (67, 18, 19), (130, 19, 34),
                                     (131, 5, 200), (4, 130, 35), (258, 258, 130), (259, 243, 146)])
def test_noalloc_divergence_at_tile_edges(storage):
    mx, my, mz = storage
    rng = np.random.default_rng(mx + my + mz)
    u = rng.standard_normal((mz, my, mx, 3))
    aj = rng.uniform(0.5, 2.0, (mz, my, mx))
    nv = np.where(rng.uniform(size=(mz, my, mx)) < 0.01, 1.4, 0.0) if mx > 5 else np.zeros((mz, my, mx))
    v, i = device(u, aj, nv)
    w, j = host(u, aj, nv)
    assert i == j and abs(v - w) <= 2.0 ** -50 * 12 * np.abs(u).max(), (storage, v, w, i, j)
    # a tie takes the smaller index, here in the last and the first tile
    u[...] = 0.0
    first = (1, 1, 1)
    for k, q, p in (first, (mz - 2, my - 2, mx - 2)):
        nv[max(k - 1, 0):k + 2, max(q - 1, 0):q + 2, max(p - 1, 0):p + 2] = 0.0
        aj[k, q, p] = 4.0
        u[k, q, p, 0] = 1.0
    v, i = device(u, aj, nv)
    w, j = host(u, aj, nv)
    assert (v, i) == (w, j), (storage, v, w, i, j)
    # no divergence anywhere: 0 at index 0
    assert device(np.zeros_like(u), aj, nv) == (0.0, 0)
    # a NaN beats every number
    u[mz - 2, my - 2, mx - 2, 0] = np.nan
    v, i = device(u, aj, nv)
    assert np.isnan(v) and i >= (mx - 2) + mx * ((my - 2) + my * (mz - 2)) - mx * my, (storage, v, i)
