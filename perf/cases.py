"""The work that users of the fractional-step library have it do, as cases
that can be timed and compared through the package's public entry points.

Every case is a whole call or a run of calls a program makes: fractional
steps of one flow (Flow_Solver) with the fields fetched at the end as a run
writes them every so many steps, the pressure solve alone (PoissonSolver_MG),
dual-time-stepping momentum (ImpRK inside Flow_Solver), a batched ensemble
(Batch.step), requests through the serving loop (Server) and Divergence on
device pointers (cv_divergence_noalloc).  Geometry is the warped, tanh-
stretched channel of curvib_old_amd.cases, with a sphere and its IB nodes
where the case names a diameter; the seed draws the perturbed initial fluxes.
"""
from __future__ import annotations

import functools

import numpy as np
import torch

from curvib_old_amd import _lib, cases, ibsearch, serving
from curvib_old_amd.solver import Batch, UserCtx

DEVICE = "cuda" if torch.cuda.is_available() else "cpu"

# the y-line preconditioner of the benchmark: 3+3 sweeps, wall-normal axis
# kept, the longest of the other axes coarsened first
YLINE = dict(smoother="yline", omega=0.9, pre_sweeps=3, post_sweeps=3, coarse_sweeps=10, restart=30, max_it=400,
             atol=0.0)
IMPRK = dict(scheme="imprk", imp_max_it=50, imp_atol=1e-7, imp_rtol=1e-4, cfl=0.2)
CHANNEL = (7, 7, 1, 1, 7, 7)
OPEN = (7, 7, 1, 1, 5, 4)       # inlet on k-, outlet on k+


def _flow(name, cells, precision, steps, re=500.0, amp=0.05, sphere=0.0, scheme="rk", bc="channel", solver="yline",
          rtol=1e-9):
    c = dict(kind="flow", cx=cells[0], cy=cells[1], cz=cells[2], precision=precision, steps=steps, re=re, amp=amp,
             sphere=sphere, scheme=scheme, bc=bc, solver=solver, rtol=rtol)
    return dict(c, name=name) if name else c


def listed():
    return [
        # Divergence checked inside a caller's own captured loop: the smallest and the largest grid
        dict(name="divergence 32x32x32", kind="divergence", cx=32, cy=32, cz=32, amp=0.05),
        dict(name="divergence 512x256x256", kind="divergence", cx=512, cy=256, cz=256, amp=0.1),
        # the smallest case of an ensemble, alone: latency of many short launches
        _flow("flow 32x32x32 mixed16", (32, 32, 32), "mixed16", 10, re=800.0, sphere=0.3),
        # a user who changes no solver option: FP64, point Jacobi, every axis coarsened
        _flow("flow 64x64x64 defaults", (64, 64, 64), "fp64", 4, re=180.0, solver="default", rtol=1e-10),
        # inlet and outlet faces, ragged sizes
        _flow("flow open 72x61x112 fp64", (72, 61, 112), "fp64", 4, amp=0.1, sphere=0.45, bc="open"),
        # the sphere channel at its configured size: production momentum scheme, then explicit RK
        _flow("imprk 256x192x192 fp64", (256, 192, 192), "fp64", 1, sphere=0.25, scheme="imprk", rtol=1e-10),
        _flow("flow 256x192x192 mixed16", (256, 192, 192), "mixed16", 6, sphere=0.25),
        # FP64 throughout, large
        _flow("flow 384x160x192 fp64", (384, 160, 192), "fp64", 4, amp=0.1, sphere=0.25),
        # the headline workload
        _flow("flow 512x256x256 mixed16", (512, 256, 256), "mixed16", 5, amp=0.1, sphere=0.25),
        # the pressure solve alone, FP32 V-cycle, ragged sizes
        dict(name="solve 200x117x136 mixed", kind="solve", cx=200, cy=117, cz=136, precision="mixed", re=500.0,
             amp=0.1, sphere=0.3, bc="channel", solver="yline", rtol=1e-9, scheme="rk"),
        # an ensemble advanced together
        dict(name="batch of 16 mixed16", kind="batch", n=16, geo=2026, precision="mixed16", steps=4, rtol=1e-9,
             solver="yline"),
        # requests through the serving loop, 4 in flight
        dict(name="serve 6 requests mixed16", kind="serve", n=6, geo=7, precision="mixed16", steps=5, slots=4,
             rtol=1e-9, solver="yline"),
    ]


def _log_uniform(rng, lo, hi):
    return lo * (hi / lo) ** rng.random()


def draw(rng):
    kind = rng.choice(("flow", "flow", "flow", "flow", "solve", "solve", "batch", "serve", "divergence"))
    if kind == "batch":
        return dict(kind="batch", n=rng.randint(4, 24), geo=rng.randint(0, 1 << 20), steps=rng.randint(1, 4), rtol=1e-9,
                    precision=rng.choice(("mixed16", "mixed16", "fp64")), solver="yline")
    if kind == "serve":
        return dict(kind="serve", n=rng.randint(2, 8), geo=rng.randint(0, 1 << 20), steps=rng.randint(2, 6),
                    slots=rng.randint(1, 6), rtol=1e-9, precision=rng.choice(("mixed16", "fp64")), solver="yline")
    if kind == "divergence":
        return dict(kind="divergence", cx=int(_log_uniform(rng, 16, 512)), cy=int(_log_uniform(rng, 16, 256)),
                    cz=int(_log_uniform(rng, 16, 256)), amp=round(rng.uniform(0.0, 0.1), 3))
    # x and z even so that multigrid can halve them (multiples of 8, 16 or 24), y any size: it is not coarsened
    size = _log_uniform(rng, 32, 256)
    snap = lambda v, q, hi: int(min(hi, max(32, q * round(v / q))))   # noqa: E731
    cx = snap(size * rng.uniform(0.8, 2.0), rng.choice((8, 16, 24)), 512)
    cy = int(min(256, max(24, size * rng.uniform(0.6, 1.0))))
    cz = snap(size * rng.uniform(0.7, 1.0), rng.choice((8, 16, 24)), 256)
    c = _flow(None, (cx, cy, cz), rng.choice(("mixed16", "mixed16", "mixed", "fp64")),
              max(1, min(8, int(2e8 / (cx * cy * cz * 6)))), re=round(rng.uniform(150.0, 1500.0)),
              amp=round(rng.uniform(0.0, 0.1), 3), sphere=rng.choice((0.0, round(rng.uniform(0.25, 0.4), 3))),
              bc=rng.choice(("channel", "channel", "open")))
    if kind == "solve":
        del c["steps"]
        return dict(c, kind="solve")
    if cx * cy * cz < 9.5e6 and rng.random() < 0.2:
        return dict(c, scheme="imprk", steps=1)
    return c


# ---------------------------------------------------------------------
# inputs: the arrays of cases.build made on the GPU (the geometry once per
# process, the perturbed fluxes from the seed)
# ---------------------------------------------------------------------
def _channel(c):
    """The ChannelCase of a single-grid case."""
    d = c.get("sphere", 0.0)
    ch = cases.ChannelCase(cells=(c["cx"], c["cy"], c["cz"]), amp=c["amp"], re=c.get("re", 500.0),
                           sphere=(0.5, 0.5, 0.5, d) if d else None)
    if c.get("bc") == "open":
        ch.bctype, ch.inlet, ch.inlet_center = OPEN, 7, (0.0, 0.5, 0.0)
    if c.get("scheme", "rk") == "rk":
        ch.dt = cases.stable_dt(ch)
    return ch


def _channels(c):
    rng = np.random.default_rng(c["geo"])
    return [serving.sample_case(rng, lo=(32, 32, 32), hi=(128, 96, 96)) for _ in range(c["n"])]


def _nodes(ch):
    """cases.node_coords on the device: (KM, JM, IM, 3)."""
    im, jm, km = ch.nodes
    f = dict(dtype=torch.float64, device=DEVICE)
    x = ch.lx * torch.arange(im, **f) / (im - 1)
    z = ch.lz * torch.arange(km, **f) / (km - 1)
    eta = torch.arange(jm, **f) / (jm - 1)
    y0 = ch.ly * 0.5 * (1.0 + torch.tanh(ch.beta * (2 * eta - 1)) / np.tanh(ch.beta))
    out = torch.empty((km, jm, im, 3), **f)
    out[..., 0] = x
    out[..., 2] = z[:, None, None]
    warp = ch.amp * torch.sin(2 * np.pi * z / ch.lz)[:, None, None] * torch.sin(2 * np.pi * x / ch.lx)
    out[..., 1] = y0[None, :, None] + warp * ((ch.ly - y0) / ch.ly)[None, :, None]
    return out


def _nvert(ch, xyz):
    """cases.nvert_field on the device: 0 fluid, 1.4 IB node, 3.4 solid."""
    mx, my, mz = ch.storage
    nv = torch.zeros((mz, my, mx), dtype=torch.float64, device=DEVICE)
    if ch.sphere is not None:
        a = xyz[1:] + xyz[:-1]
        a = a[:, 1:] + a[:, :-1]
        cent = 0.125 * (a[:, :, 1:] + a[:, :, :-1])
        c0 = torch.tensor(ch.sphere[:3], dtype=torch.float64, device=DEVICE)
        core = ((cent - c0) ** 2).sum(-1) < (0.5 * ch.sphere[3]) ** 2
        near = torch.nn.functional.max_pool3d(core[None, None].float(), 3, 1, 1)[0, 0] > 0
        nv[1:-1, 1:-1, 1:-1][near] = 1.4
        nv[1:-1, 1:-1, 1:-1][core] = 3.4
    if ch.bctype[0] == 7:
        nv[:, :, 0], nv[:, :, -1] = nv[:, :, -2].clone(), nv[:, :, 1].clone()
    if ch.bctype[4] == 7:
        nv[0], nv[-1] = nv[-2].clone(), nv[1].clone()
    return nv


@functools.lru_cache(maxsize=48)
def _geometry(key):
    """Node coordinates, nvert and IB records of one channel as host arrays."""
    ch = cases.ChannelCase(**dict(key))
    xyz = _nodes(ch)
    nv = _nvert(ch, xyz).cpu().numpy()
    xyz = xyz.cpu().numpy()
    return xyz, nv, ibsearch.sphere_ib_nodes(ch, xyz, nv) if ch.sphere else None


def _geo(ch):
    return _geometry(tuple(sorted((k, getattr(ch, k)) for k in ("cells", "beta", "amp", "sphere", "bctype"))))


def _flux(ch, xyz, nvert, seed):
    """cases.initial_ucont on the device: the parabolic profile with every
    face velocity component perturbed by up to ch.pert, dotted with the face
    areas; no flux through walls and body faces."""
    mx, my, mz = ch.storage
    gen = torch.Generator(device=DEVICE).manual_seed(int(seed))
    c = torch.zeros((mz, my, mx, 3), dtype=torch.float64, device=DEVICE)
    c[:-1, :-1, :-1] = torch.as_tensor(xyz, device=DEVICE)
    uc = torch.zeros_like(c)
    # per axis: corners a b (axis +t) and c d of the face's quadrilateral in cyclic order
    for d in range(3):
        t, s = (d + 1) % 3, (d + 2) % 3                      # tangential axes, right-handed

        def corner(dt, ds):
            sl = [None] * 3                                  # x, y, z slices
            for ax, m in ((0, mx), (1, my), (2, mz)):
                low = 0 if ax == d else 1                    # the face index starts at 0 along its own axis
                off = dt if ax == t else ds if ax == s else 0
                sl[ax] = slice(low - off, m - 1 - off)
            return c[sl[2], sl[1], sl[0]]
        p, q, r, o = corner(0, 0), corner(1, 0), corner(0, 1), corner(1, 1)
        area = torch.linalg.cross(0.5 * (p + r - q - o), 0.5 * (p + q - r - o))
        y = 0.25 * (p + q + r + o)[..., 1] / ch.ly
        v = ch.pert * (2.0 * torch.rand(area.shape, generator=gen, dtype=torch.float64, device=DEVICE) - 1.0)
        v[..., 2] += 1.5 * (1.0 - (2.0 * y - 1.0) ** 2)
        lo = [0 if ax == d else 1 for ax in range(3)]
        uc[lo[2]:mz - 1, lo[1]:my - 1, lo[0]:mx - 1, d] = (v * area).sum(-1)
        del p, q, r, o, area, y, v
    bc = ch.bctype
    solid = torch.as_tensor(nvert, device=DEVICE) > 0.1
    for d, (ax, m) in enumerate(((2, mx), (1, my), (0, mz))):
        u = uc[..., d]
        if bc[2 * d] == 1:
            u.select(ax, 0).zero_()
        if bc[2 * d + 1] == 1:
            u.select(ax, m - 2).zero_()
        u.narrow(ax, 0, m - 1)[solid.narrow(ax, 0, m - 1) | solid.narrow(ax, 1, m - 1)] = 0.0
        if bc[2 * d] == 7:
            u.select(ax, 0).copy_(u.select(ax, m - 2))
    return uc


def _arrays(ch, seed):
    xyz, nv, ib = _geo(ch)
    return xyz, nv, _flux(ch, xyz, nv, seed).cpu().numpy(), ib


def _context(c, ch, seed):
    xyz, nv, uc, ib = _arrays(ch, seed)
    if c["solver"] == "default":
        u = UserCtx(ch.nodes, ch.bctype, 4, ch.re, ch.dt)
        u.set_solver(precision=c["precision"], rtol=c["rtol"], max_it=400)
    else:
        u = UserCtx(ch.nodes, ch.bctype, serving.levels_for(ch.cells), ch.re, ch.dt, semi=serving.SEMI,
                    coarsen_auto=serving.COARSEN_AUTO, inlet=ch.inlet, inlet_center=ch.inlet_center)
        u.set_solver(precision=c["precision"], rtol=c["rtol"], **YLINE)
    if c.get("scheme") == "imprk":
        u.set_momentum(**IMPRK)
    u.set_grid(xyz)
    u.set_nvert(nv)
    if ib is not None:
        u.set_ib_nodes(*ib)
    u.put("ucont", uc)
    return u


def _fields(u):
    return [u.get("p"), u.get("ucont")]


def prepare(case, seed):
    c = case
    if c["kind"] == "divergence":
        ch = _channel(c)
        xyz, nv, _ = _geo(ch)
        uc = _flux(ch, xyz, nv, seed)
        y = torch.as_tensor(xyz[..., 1], device=DEVICE)
        dy = y[:, 1:] - y[:, :-1]
        dy = dy[1:] + dy[:-1]
        aj = torch.zeros(uc.shape[:3], dtype=torch.float64, device=DEVICE)
        aj[1:-1, 1:-1, 1:-1] = ch.cells[0] * ch.cells[2] / (0.25 * (dy[:, :, 1:] + dy[:, :, :-1]))
        return dict(case=c, ucont=uc, aj=aj, nvert=torch.as_tensor(nv, device=DEVICE),
                    out=torch.zeros(2, dtype=torch.float64, device=DEVICE))
    if c["kind"] in ("flow", "solve"):
        return dict(case=c, ctx=_context(c, _channel(c), seed))
    chs = _channels(c)
    if c["kind"] == "batch":
        ctxs = [_context(c, ch, seed + 1000 * q) for q, ch in enumerate(chs)]
        return dict(case=c, ctxs=ctxs, batch=_Batch(ctxs))
    return dict(case=c, server=serving.Server(budget_bytes=100e9, slots=c["slots"]),
                requests=[(ch, _arrays(ch, seed + 1000 * q)) for q, ch in enumerate(chs)])


class _Batch(Batch):
    """A batch that goes before its contexts when the state is dropped."""

    def __del__(self):
        self.close()
        for u in self.ctxs:
            u.close()


def run(state):
    c = state["case"]
    if c["kind"] == "divergence":
        mz, my, mx = state["aj"].shape
        _lib.check(_lib.load().cv_divergence_noalloc(
            0, state["ucont"].data_ptr(), state["aj"].data_ptr(), state["nvert"].data_ptr(), mx, my, mz,
            torch.cuda.current_stream().cuda_stream, state["out"].data_ptr()), "cv_divergence_noalloc")
        return state["out"]
    if c["kind"] == "solve":
        state["ctx"].PoissonSolver_MG()
        return state["ctx"].get("phi")
    if c["kind"] == "flow":
        for _ in range(c["steps"]):
            state["ctx"].Flow_Solver()
        return _fields(state["ctx"])
    if c["kind"] == "batch":
        for _ in range(c["steps"]):
            state["batch"].step()
        return [_fields(u) for u in state["ctxs"]]
    srv, ids, out = state["server"], [], []
    for ch, arrays in state["requests"]:
        ids.append(srv.submit(ch, arrays, c["steps"], precision=c["precision"], rtol=c["rtol"], **YLINE))
    for (ch, _), cid in zip(state["requests"], ids):
        rc, info = srv.wait(cid)
        _lib.check(rc, f"request {cid}")
        mx, my, mz = ch.storage
        out.append([srv.fetch(cid, "p", (mz, my, mx)), srv.fetch(cid, "ucont", (mz, my, mx, 3))])
        srv.release(cid)
    return out


def work(case):
    """Per storage point: Divergence reads 5 values.  A solve reads the
    operator (9 coefficients, 1/J, nvert) and the fluxes and writes phi; a
    step also reads the 40 metric values and reads and writes Ucont, Ucat
    and p.  Operations: about 900 per point for one momentum right-hand side
    (four a step, or four per pseudo-time iteration of which at least ten
    run) and 1500 per multigrid iteration of which about ten run."""
    c = case
    if c["kind"] == "divergence":
        n = (c["cx"] + 2) * (c["cy"] + 2) * (c["cz"] + 2)
        return {"bytes": 40.0 * n, "flops": 8.0 * n}
    chs = [_channel(c)] if c["kind"] in ("flow", "solve") else _channels(c)
    n = float(sum(np.prod(ch.storage) for ch in chs))
    if c["kind"] == "solve":
        return {"bytes": n * 8 * (11 + 3 + 1), "flops": n * 10 * 1500}
    rhs = 40 if c.get("scheme") == "imprk" else 4
    return {"bytes": n * c["steps"] * 8 * (40 + 11 + 2 * 7), "flops": n * c["steps"] * (rhs * 900 + 10 * 1500)}


def exact(case, seed):
    """The largest divergence and its first storage index.  None for the
    flows and solves: their values come out of an iterative solution that
    plain 64-bit torch would not reach within the time allowed."""
    if case["kind"] != "divergence":
        return None
    s = prepare(case, seed)
    u, aj, nv = s["ucont"], s["aj"], s["nvert"]
    i = slice(1, -1)
    lo = slice(0, -2)
    div = torch.zeros_like(aj)
    div[i, i, i] = ((u[i, i, i, 0] - u[i, i, lo, 0] + u[i, i, i, 1] - u[i, lo, i, 1] + u[i, i, i, 2] - u[lo, i, i, 2])
                    * aj[i, i, i]).abs()
    hi = slice(2, None)
    near = nv[i, i, i] + nv[hi, i, i] + nv[lo, i, i] + nv[i, hi, i] + nv[i, lo, i] + nv[i, i, hi] + nv[i, i, lo]
    div[i, i, i][near > 0.1] = 0.0
    q = int(div.reshape(-1).argmax())
    return torch.tensor([float(div.reshape(-1)[q]), float(q)], dtype=torch.float64)
