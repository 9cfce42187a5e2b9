"""The work that users of hydro_amd have it do, as cases to be measured.

Every case goes through the package's public entry points, the way bench.py,
the drop-in driver and the tests use them.  Six kinds:

* solve   -- one grid: a blast set up on the GPU, `steps` steps of the device
             time loop with the dt of each step, the final state downloaded;
             or, with output "image", the density image of it.
* restart -- one grid continued from a state in host memory (a checkpoint): an
             upload, `steps` steps, a download.
* driver  -- the host time loop of the drop-in call surface: compute_deltat on
             even steps, one godunov call a step, then the download.
* batch   -- many uneven grids advanced together, every state downloaded.
* serve   -- a set of requests put to the continuous-batching server, which is
             pumped until all are done, and their results.
* deltat  -- the allocation-free CFL step on a state the caller has on the GPU.

Blasts, energies and gammas are drawn as in hydro_amd/workloads.py; the
uploaded states are smooth and move everywhere, so that every cell's Riemann
problem is a real one.  Outputs are whole: states, dt sequences, times, images.
"""
from __future__ import annotations

import math

import numpy as np
import torch

import hydro_amd

FORMS = {"fp64": hydro_amd.FP64, "fast": hydro_amd.FP64_FAST, "mixed": hydro_amd.MIXED}
BYTES = {"fp64": 8, "fast": 8, "mixed": 4}  # a stored value


def listed():
    return [
        # the smallest call: dt of a deck-sized state that a caller's own program holds
        dict(name="deltat_250x125", kind="deltat", nx=250, ny=125),
        # the 250x125 corner deck: 100 steps, latency alone
        dict(name="solve_250x125_fp64", kind="solve", nx=250, ny=125, form="fp64", steps=100,
             output="state"),
        # the drop-in driver's host loop on the 500x500 deck
        dict(name="driver_500x500_fp64", kind="driver", nx=500, ny=500, form="fp64", steps=40),
        # a checkpoint of an odd-sized flow that moves everywhere, continued
        dict(name="restart_1021x767_fp64", kind="restart", nx=1021, ny=767, form="fp64", steps=60,
             boundary=3, slope=1.0),
        # the same in the mixed form, reflecting walls, a steeper limiter
        dict(name="restart_1531x1200_mixed", kind="restart", nx=1531, ny=1200, form="mixed",
             steps=60, boundary=1, slope=2.0),
        # an ordinary production grid, bit for bit
        dict(name="solve_4099x3001_fp64", kind="solve", nx=4099, ny=3001, form="fp64", steps=60,
             output="state"),
        # one of eight row bands of the headline grid, an image every 50 steps
        dict(name="image_8192x1024_fast", kind="solve", nx=8192, ny=1024, form="fast", steps=50,
             output="image"),
        # the headline grid and length, in the form it is quoted in
        dict(name="solve_8192x8192_fast", kind="solve", nx=8192, ny=8192, form="fast", steps=200,
             output="state"),
        # the same grid in the mixed form
        dict(name="solve_8192x8192_mixed", kind="solve", nx=8192, ny=8192, form="mixed", steps=200,
             output="state"),
        # batched uneven grids, 100 steps each
        dict(name="batch_60_fp64", kind="batch", n=60, lo=64, hi=1024, form="fp64", steps=100),
        dict(name="batch_60_fast", kind="batch", n=60, lo=64, hi=1024, form="fast", steps=100),
        # the serving mix: everything queued at once
        dict(name="serve_24_mixed", kind="serve", n=24, lo=128, hi=4096, form="mixed", steps=200),
    ]


def _log(rng, lo, hi):
    return int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))


def draw(rng):
    kind = rng.choice(["solve", "solve", "restart", "driver", "batch", "serve", "deltat"])
    form = rng.choice(["fp64", "fast", "mixed"])
    if kind == "deltat":
        return dict(kind=kind, nx=_log(rng, 48, 4096), ny=_log(rng, 48, 4096))
    if kind in ("batch", "serve"):
        lo = _log(rng, 48, 200)
        hi = _log(rng, 2 * lo, 1024 if kind == "batch" else 3000)
        return dict(kind=kind, n=rng.randint(5, 60 if kind == "batch" else 24), lo=lo, hi=hi,
                    form="mixed" if kind == "serve" else form, steps=rng.randint(20, 100))
    top = 8192 if kind == "solve" else 2000
    c = dict(kind=kind, nx=_log(rng, 40, top), ny=_log(rng, 40, top), form=form,
             steps=rng.randint(10, 100 if kind == "solve" else 60))
    if kind == "solve":
        c["output"] = rng.choice(["state", "state", "image"])
    elif kind == "restart":
        c["boundary"] = rng.choice([1, 3])
        c["slope"] = rng.choice([1.0, 2.0])
    return c


# ---- inputs ------------------------------------------------------------------------


def _params(case, gamma, nx=None, ny=None, nstepmax=2**31 - 1, tend=1e30):
    nx, ny = nx or case["nx"], ny or case["ny"]
    b = case.get("boundary", 1)
    return hydro_amd.Params(
        nx=nx, ny=ny, dx=1.0 / max(nx, ny), gamma=gamma, courant_factor=0.8, niter_riemann=10,
        iorder=2, slope_type=case.get("slope", 1.0), tend=tend, nstepmax=nstepmax,
        precision=FORMS[case.get("form", "fp64")], boundary_left=b, boundary_right=b,
        boundary_down=b, boundary_up=b)


def _blast(rng, nx, ny):
    dx = 1.0 / max(nx, ny)
    return (int(rng.integers(0, nx)), int(rng.integers(0, ny)),
            float(rng.uniform(0.1, 10.0)) / dx / dx)


def _smooth(rng, p):
    """Densities around 1, subsonic and mildly supersonic speeds, pressures around 1."""
    x = (np.arange(p.nx + 4) - 1.5) / p.nx
    y = (np.arange(p.ny + 4) - 1.5) / p.ny

    def waves(amp):
        f = np.zeros((p.ny + 4, p.nx + 4))
        for _ in range(4):
            kx, ky = rng.integers(1, 7, 2)
            f += np.outer(np.cos(2 * np.pi * ky * y + rng.uniform(0, 6.28)),
                          np.cos(2 * np.pi * kx * x + rng.uniform(0, 6.28)))
        return amp / 4 * f

    rho, u, v, pr = np.exp(waves(0.8)), waves(2.0), waves(2.0), np.exp(waves(0.8))
    return np.ascontiguousarray(
        np.stack([rho, rho * u, rho * v, pr / (p.gamma - 1) + 0.5 * rho * (u * u + v * v)]))


def _many(case, rng):
    """The grids of a batch or a set of requests: (params, bx, by, e) each."""
    out = []
    for _ in range(case["n"]):
        side = int(np.exp(rng.uniform(np.log(case["lo"]), np.log(case["hi"]))))
        side = max(case["lo"], min(case["hi"], side))
        p = _params(case, float(rng.uniform(1.3, 1.67)), side, side, nstepmax=case["steps"],
                    tend=0.1 if case["kind"] == "serve" else 1e30)
        out.append((p, *_blast(rng, side, side)))
    return out


def _inputs(case, seed):
    rng = np.random.default_rng(seed)
    kind = case["kind"]
    if kind in ("batch", "serve"):
        # the grids' sizes are the case's own; blasts and gammas are the seed's
        sizes = _many(case, np.random.default_rng(case["n"] * 131071 + case["hi"]))
        runs = []
        for q, *_ in sizes:
            p = _params(case, float(rng.uniform(1.3, 1.67)), q.nx, q.ny, q.nstepmax, q.tend)
            runs.append((p, *_blast(rng, p.nx, p.ny)))
        return runs
    p = _params(case, float(rng.uniform(1.3, 1.67)))
    if kind in ("restart", "deltat"):
        return p, _smooth(rng, p)
    return (p, *_blast(rng, p.nx, p.ny))


def prepare(case, seed):
    kind, inp = case["kind"], _inputs(case, seed)
    s = dict(case=case, kind=kind)
    if kind == "deltat":
        p, u = inp
        s.update(p=p, u=torch.from_numpy(u).cuda(),
                 dt=torch.zeros(1, dtype=torch.float64, device="cuda"))
        torch.cuda.synchronize()
    elif kind == "batch":
        b = hydro_amd.Batch(FORMS[case["form"]])
        s.update(batch=b, runs=inp, ids=[b.add(r[0]) for r in inp])
        b.sync()
    elif kind == "serve":
        srv = hydro_amd.Server(precision=FORMS[case["form"]], budget_bytes=100 * 10**9,
                               chunk_steps=20, keep_results=True)
        srv.reserve_results(sum(16 * (r[0].nx + 4) * (r[0].ny + 4) + 256 for r in inp))
        s.update(server=srv, runs=inp)
    else:
        s.update(grid=hydro_amd.Grid(inp[0]), inp=inp)
    return s


def run(s):
    case, kind = s["case"], s["kind"]
    if kind == "deltat":
        hydro_amd.compute_deltat_noalloc(s["p"], s["u"].data_ptr(), s["dt"].data_ptr(),
                                         torch.cuda.current_stream().cuda_stream)
        return s["dt"]
    if kind == "batch":
        b = s["batch"]
        for i, (_, bx, by, e) in zip(s["ids"], s["runs"]):
            b.init_blast(i, bx, by, e)
        b.run(case["steps"])
        q = b.query()
        return {"t": np.array([q[i][0] for i in s["ids"]]),
                "u": [b.download(i) for i in s["ids"]]}
    if kind == "serve":
        srv = s["server"]
        ids = [srv.submit(*r) for r in s["runs"]]
        while srv.pump() > 0:
            pass
        out = {"t": np.array([srv.info(i)[4] for i in ids]), "u": [srv.result(i) for i in ids]}
        for i in ids:
            srv.release(i)
        return out
    g = s["grid"]
    if kind == "restart":
        g.upload(s["inp"][1])
        g.set_state(0.0, 0, 0.0)
        dts = g.run(case["steps"])
        return {"dt": dts, "u": g.download()}
    _, bx, by, e = s["inp"]
    g.init_blast(bx, by, e)
    if kind == "driver":
        dts, dt = [], 0.0
        for n in range(case["steps"]):
            if n % 2 == 0:
                dt = g.compute_deltat()
                if n == 0:
                    dt /= 2.0
            g.godunov(1 if n % 2 == 0 else 2, dt)
            dts.append(dt)
        return {"dt": np.array(dts), "u": g.download()}
    dts = g.run(case["steps"])
    return {"dt": dts, "image": g.image(1000)} if case["output"] == "image" else \
        {"dt": dts, "u": g.download()}


def work(case):
    """A step reads a cell's four values and writes them once (the state is far
    larger than the chip holds, or small enough not to matter) and takes about
    600 operations of it; a state handed out is 32 bytes a cell."""
    kind = case["kind"]
    if kind == "deltat":
        n = case["nx"] * case["ny"]
        return {"bytes": 32.0 * n, "flops": 25.0 * n}
    if kind in ("batch", "serve"):
        n = sum(r[0].nx * r[0].ny for r in _inputs(case, 0))
    else:
        n = case["nx"] * case["ny"]
    outs = n * 32.0 if case.get("output") != "image" else 0.0
    if kind == "restart":
        outs *= 2
    return {"bytes": 8.0 * BYTES[case["form"]] * n * case["steps"] + outs,
            "flops": 600.0 * n * case["steps"]}


# ---- the same in plain torch, 64 bits ------------------------------------------------


def _prim(u, p):
    r = torch.clamp(u[0], min=p.smallr)
    vx, vy = u[1] / r, u[2] / r
    e = u[3] / r - 0.5 * (vx * vx + vy * vy)
    pr = torch.maximum((p.gamma - 1.0) * r * e, r * (p.smallc**2 / p.gamma))
    return r, vx, vy, pr, torch.sqrt(p.gamma * pr / r)


def _deltat(u, p):
    _, vx, vy, _, c = _prim(u[:, 2:-2, 2:-2], p)
    top = max(float((c + vx.abs()).max()), float((c + vy.abs()).max()), p.smallc)
    return p.courant_factor * p.dx / top


def _ghosts(u, idim, p):
    """Two ghost layers of the lines along direction idim (types 1 and 3)."""
    n = p.nx if idim == 1 else p.ny
    line = (lambda k: u[:, 2:-2, k]) if idim == 1 else (lambda k: u[:, k, 2:-2])
    lo, hi = ((p.boundary_left, p.boundary_right) if idim == 1
              else (p.boundary_down, p.boundary_up))
    for g, typ in ((0, lo), (1, lo), (n + 2, hi), (n + 3, hi)):
        mirror = typ == 1
        k = (3 - g if g < 2 else 2 * n + 3 - g) if mirror else (n + g if g < 2 else g - n)
        line(g)[:] = line(k)
        if mirror:
            line(g)[idim] *= -1.0


def _riemann(ql, qr, p):
    smallp, g6 = p.smallc**2 / p.gamma, (p.gamma + 1.0) / (2.0 * p.gamma)
    rl, rr = torch.clamp(ql[0], min=p.smallr), torch.clamp(qr[0], min=p.smallr)
    ul, ur = ql[1], qr[1]
    pl, pr = torch.maximum(ql[3], rl * smallp), torch.maximum(qr[3], rr * smallp)
    cl, cr = p.gamma * pl * rl, p.gamma * pr * rr
    wl, wr = torch.sqrt(cl), torch.sqrt(cr)
    ps = torch.clamp((wr * pl + wl * pr + wl * wr * (ul - ur)) / (wl + wr), min=0.0)
    going = torch.ones_like(ps, dtype=torch.bool)
    for _ in range(p.niter_riemann):
        a = torch.sqrt(cl * (1.0 + g6 * (ps - pl) / pl))
        b = torch.sqrt(cr * (1.0 + g6 * (ps - pr) / pr))
        fl, fr = 2.0 * a * (a * a) / (a * a + cl), 2.0 * b * (b * b) / (b * b + cr)
        d = fr * fl / (fr + fl) * ((ul - (ps - pl) / a) - (ur + (ps - pr) / b))
        d = torch.where(going, torch.maximum(d, -ps), torch.zeros_like(ps))
        ps = ps + d
        going &= (d / (ps + p.smallr * smallp)).abs() > 1e-6
        if not bool(going.any()):
            break
    wr = torch.sqrt(cr * (1.0 + g6 * (ps - pr) / pr))
    wl = torch.sqrt(cl * (1.0 + g6 * (ps - pl) / pl))
    us = 0.5 * (ul + (pl - ps) / wl + ur - (pr - ps) / wr)
    left = us > 0
    sg = torch.where(left, 1.0, -1.0).to(ps.dtype)
    ro, uo, po, wo, vo = (torch.where(left, a, b) for a, b in
                          ((rl, rr), (ul, ur), (pl, pr), (wl, wr), (ql[2], qr[2])))
    co = torch.clamp(torch.sqrt((p.gamma * po / ro).abs()), min=p.smallc)
    rs = torch.clamp(ro / (1.0 + ro * (po - ps) / (wo * wo)), min=p.smallr)
    cs = torch.clamp(torch.sqrt((p.gamma * ps / rs).abs()), min=p.smallc)
    shock = ps >= po
    out, inn, ush = co - sg * uo, cs - sg * us, wo / ro - sg * uo
    out, inn = torch.where(shock, ush, out), torch.where(shock, ush, inn)
    frac = (1.0 + (out + inn) / torch.maximum(out - inn, p.smallc + (out + inn).abs())) * 0.5
    frac = torch.clamp(frac, 0.0, 1.0)
    frac = torch.where(inn > 0.0, torch.ones_like(frac), frac)
    frac = torch.where(out < 0.0, torch.zeros_like(frac), frac)
    # (weights of exactly 0 and 1 give the outer and the star state themselves)
    r, u, q = (frac * s + (1.0 - frac) * o for s, o in ((rs, ro), (us, uo), (ps, po)))
    m = r * u
    en = q / (p.gamma - 1.0) + 0.5 * r * (u * u + vo * vo)
    return m, m * u + q, m * vo, u * (en + q)


def _sweep(u, idim, dt, p):
    """One direction over the interior lines; lines run along the last axis."""
    w = u[:, 2:-2, :] if idim == 1 else u[[0, 2, 1, 3]][:, :, 2:-2].transpose(1, 2)
    w = w.contiguous()
    k, st = dt / p.dx, p.slope_type
    r, un, ut, pr, c = _prim(w, p)
    dq = []
    for a in (r, un, ut, pr):
        dl, dr = st * (a[:, 1:-1] - a[:, :-2]), st * (a[:, 2:] - a[:, 1:-1])
        dc = 0.5 * (dl + dr) / st
        lim = torch.where(dl * dr <= 0.0, torch.zeros_like(dl), torch.minimum(dl.abs(), dr.abs()))
        dq.append(torch.sign(dc) * torch.minimum(lim, dc.abs()))
    r, un, ut, pr, c = (a[:, 1:-1] for a in (r, un, ut, pr, c))
    dr, du, dv, dp = dq
    am, ap = 0.5 * (dp / (r * c) - du) * (r / c), 0.5 * (dp / (r * c) + du) * (r / c)
    a0 = dr - dp / (c * c)
    side = []
    for one in (-1.0, 1.0):  # the right face (seen from inside), the left face
        m, q_, z = -0.5 * ((un - c) * k + one), -0.5 * ((un + c) * k + one), -0.5 * (un * k + one)
        side.append((r + (q_ * ap + m * am + z * a0), un + (q_ * ap - m * am) * (c / r),
                     ut + z * dv, pr + (q_ * ap + m * am) * (c * c)))
    f = _riemann([a[:, :-1] for a in side[0]], [a[:, 1:] for a in side[1]], p)
    new = [w[v][:, 2:-2] + (f[v][:, :-1] - f[v][:, 1:]) * k for v in range(4)]
    if idim == 1:
        for v in range(4):
            u[v, 2:-2, 2:-2] = new[v]
    else:
        for v, g in enumerate((0, 2, 1, 3)):
            u[g, 2:-2, 2:-2] = new[v].transpose(0, 1)


def _advance(u, p, steps, tend=1e30):
    t, dt, dts = 0.0, 0.0, []
    for n in range(steps):
        if not t < tend:
            break
        if n % 2 == 0:
            dt = _deltat(u, p) * (0.5 if n == 0 else 1.0)
        for idim in ((1, 2) if n % 2 == 0 else (2, 1)):
            _ghosts(u, idim, p)
            _sweep(u, idim, dt, p)
        dts.append(dt)
        t += dt
    return dts, t


def _blast_state(p, bx, by, e, dev):
    u = torch.zeros(p.shape(), dtype=torch.float64, device=dev)
    u[0, 2:-2, 2:-2] = 1.0
    u[3, 2:-2, 2:-2] = 1e-5
    u[3, by + 2, bx + 2] = e
    return u


def exact(case, seed):
    dev = "cuda" if torch.cuda.is_available() else "cpu"
    room = 6e8 if dev == "cuda" else 4e6  # cell-steps that fit the time
    kind, inp = case["kind"], _inputs(case, seed)
    if kind == "deltat":
        p, u = inp
        return np.array([_deltat(torch.from_numpy(u).to(dev), p)])
    if kind in ("batch", "serve"):
        ts, us = [], []
        for p, bx, by, e in inp:  # the first few small ones
            n = p.nx * p.ny * case["steps"]
            if len([u for u in us if u is not None]) >= 3 or n > 0.1 * room:
                us.append(None)
                continue
            u = _blast_state(p, bx, by, e, dev)
            ts.append(_advance(u, p, case["steps"], p.tend)[1])
            us.append(u.cpu().numpy())
        return {"t": None, "u": us}
    if case["nx"] * case["ny"] * case["steps"] > room:
        return None
    if kind == "restart":
        p, u = inp[0], torch.from_numpy(inp[1]).to(dev)
    else:
        p, *b = inp
        u = _blast_state(p, *b, dev)
    dts, _ = _advance(u, p, case["steps"])
    return {"dt": np.array(dts), "image": None} if case.get("output") == "image" else \
        {"dt": np.array(dts), "u": u.cpu().numpy()}
