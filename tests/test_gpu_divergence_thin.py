"""cv_divergence_noalloc on grids of few columns, rows or planes and on both sides
of the sizes where a lane takes 1, 8 and 16 planes, against the same expression
in torch, and its time on thin grids against a cube's.

The value is one rounding away from torch's at most where the compiler fuses the
last product (2^-50 of the largest term); the index is exact, the inputs keeping
the largest value apart.  A thin grid moves the bytes of the cube with as many
points, so it takes about its time: three times that is the limit, where lanes
left idle by the shape cost eight and thirty-four times."""
import ctypes as C
import time

import pytest

from curvib_old_amd import _lib

pytestmark = pytest.mark.gpu
torch = pytest.importorskip("torch")


def fields(storage, seed):
    mx, my, mz = storage
    g = torch.Generator(device="cuda").manual_seed(seed)
    u = torch.rand((mz, my, mx, 3), dtype=torch.float64, device="cuda", generator=g) - 0.5
    aj = torch.rand((mz, my, mx), dtype=torch.float64, device="cuda", generator=g) + 0.5
    nv = 1.4 * (torch.rand((mz, my, mx), device="cuda", generator=g) < 0.003).double()
    return u, aj, nv


def caller(u, aj, nv):
    mz, my, mx = aj.shape
    out = torch.full((2,), -7.0, dtype=torch.float64, device="cuda")
    args = (0, *(C.c_void_p(a.data_ptr()) for a in (u, aj, nv)), mx, my, mz,
            C.c_void_p(torch.cuda.current_stream().cuda_stream), C.c_void_p(out.data_ptr()))
    return out, lambda: _lib.check(_lib.load().cv_divergence_noalloc(*args), "cv_divergence_noalloc")


# 6291456 interior points are the most that take one plane a lane: (130, 194, 258)
# below holds 128 x 192 x 256; 1030 x 1030 columns the fewest of 17 planes that take 16
@pytest.mark.parametrize("storage", [(3, 3, 5000), (5000, 3, 3), (3, 5000, 3), (3, 300, 401), (4, 257, 300), (300, 3, 301),
                                     (7, 1025, 90), (33, 31, 999), (1001, 4, 57), (255, 513, 5), (130, 194, 258),
                                     (130, 194, 259), (3, 3001, 2500), (2500, 3001, 3), (1030, 1030, 18),
                                     (1030, 1030, 19), (1020, 1020, 19)])
def test_thin_grids_match_torch(storage):
    u, aj, nv = fields(storage, sum(storage))
    c, lo, hi = slice(1, -1), slice(0, -2), slice(2, None)
    d = torch.zeros_like(aj)
    d[c, c, c] = ((u[c, c, c, 0] - u[c, c, lo, 0] + u[c, c, c, 1] - u[c, lo, c, 1] + u[c, c, c, 2] - u[lo, c, c, 2])
                  * aj[c, c, c]).abs()
    near = nv[c, c, c] + nv[hi, c, c] + nv[lo, c, c] + nv[c, hi, c] + nv[c, lo, c] + nv[c, c, hi] + nv[c, c, lo]
    d[c, c, c][near > 0.1] = 0.0
    i = int(d.argmax())
    w = float(d.reshape(-1)[i])
    out, call = caller(u, aj, nv)
    call()
    v, j = out.tolist()
    assert int(j) == i and abs(v - w) <= 2.0 ** -50 * 6, (storage, v, w, j, i)


def best_us(storage, calls):
    _, call = caller(*fields(storage, 5))
    best = 1e30
    for _ in range(6):
        torch.cuda.synchronize()
        t = time.perf_counter()
        for _ in range(calls):
            call()
        torch.cuda.synchronize()
        best = min(best, 1e6 * (time.perf_counter() - t) / calls)
    return best


@pytest.mark.parametrize("thin,cube", [((4, 1000, 1000), 159), ((3, 3, 100000), 97), ((34, 300, 300), 145),
                                       ((1000, 3, 1000), 144)])
def test_thin_grids_take_the_time_of_a_cube(thin, cube):
    a, b = best_us(thin, 60), best_us((cube,) * 3, 60)
    print(f"divergence {thin}: {a:.1f} us, {cube}^3: {b:.1f} us", flush=True)
    assert a < 3 * b, (thin, a, b)
