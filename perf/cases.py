"""What the performance of this framework is measured on.

A case is one piece of a simulation as a user's program runs it through
ctca_amd.emg: a few time steps of the electrostatic or the electromagnetic
loop with the fields on the device and a diagnostic read-out, the drop-in step
of a host field solver, a restart (upload, steps, download), and the reverse
step of the differentiable window.  `form` is the context's precision form.

`exact` restates the same step in 64-bit torch (the scheme of the reference:
trilinear gather, Buneman-Boris, CIC charge, zigzag current, Yee update,
7-point spectral Poisson), with nothing of this package.
"""
import math

import numpy as np
import torch

from ctca_amd import emg

# particles per chunk of the 64-bit restatement
CHUNK = 1 << 24


# --------------------------------------------------------------------- cases
def listed():
    return [
        # One ES step of a 16^3 test problem with its diagnostics: launches
        # and read-out latency are all there is.
        dict(name="es16_fp32", kind="es", form="fp32", nx=16, ny=16, nz=16, ppc=16.0, steps=1,
             wc=0.0, ramp=0.0),
        # The plain ES configuration (32^3, 2 x 524,288 particles) in the
        # drop-in form, a diagnostic every 10 steps.
        dict(name="es32_fp64", kind="es", form="fp64", nx=32, ny=32, nz=32, ppc=16.0, steps=10,
             wc=0.0, ramp=0.0),
        # The same in the FP32 form.
        dict(name="es32_fp32", kind="es", form="fp32", nx=32, ny=32, nz=32, ppc=16.0, steps=10,
             wc=0.0, ramp=0.0),
        # A production box whose axes are no multiples of anything.
        dict(name="es_ragged_fp32", kind="es", form="fp32", nx=90, ny=70, nz=51, ppc=20.0,
             steps=8, wc=0.2, ramp=0.0),
        # The magnetised scale-up (268,435,456 particles): the headline
        # workload, here with its field solve, in both forms.
        dict(name="mag128_fp32", kind="es", form="fp32", nx=128, ny=128, nz=128, ppc=64.0,
             steps=4, wc=0.5, ramp=0.0),
        dict(name="mag128_fp64", kind="es", form="fp64", nx=128, ny=128, nz=128, ppc=64.0,
             steps=4, wc=0.5, ramp=0.0),
        # The exp(z) density ramp at 8 particles per cell and species: sparse
        # layers and dense ones.
        dict(name="ramp_fp32", kind="es", form="fp32", nx=256, ny=256, nz=64, ppc=8.0, steps=12,
             wc=0.2, ramp=100.0),
        # The EM two-stream (32 background + 3.2 beam electrons per cell),
        # fields on the device, in both forms.
        dict(name="em_fp32", kind="em", form="fp32", nx=128, ny=128, nz=64, ppc=32.0, steps=20,
             wc=0.0, ramp=0.0),
        dict(name="em_fp64", kind="em", form="fp64", nx=128, ny=64, nz=64, ppc=32.0, steps=10,
             wc=0.0, ramp=0.0),
        # The drop-in step under a host field solver: eb in, rho with its
        # ghost planes out.
        dict(name="host64_fp64", kind="host", form="fp64", nx=64, ny=64, nz=64, ppc=16.0, steps=1,
             wc=0.5, ramp=0.0),
        # A continued job: records in, steps, records out (in upload order).
        dict(name="restart_fp64", kind="restart", form="fp64", nx=48, ny=48, nz=48, ppc=8.0,
             steps=4, wc=0.5, ramp=0.0),
        # Two reverse steps of the 64^3 differentiable window (8.8M particles).
        dict(name="adjoint64_fp64", kind="adjoint", form="fp64", nx=64, ny=64, nz=64, ppc=32.0,
             steps=2, wc=0.1, ramp=0.0),
    ]


def draw(rng):
    """One more case of these ranges."""
    kind = rng.choice(["es", "es", "es", "em", "em", "host", "restart", "adjoint"])
    form = "fp64" if kind == "adjoint" else rng.choice(["fp32", "fp64"])
    most = {"es": 6.0e7, "em": 4.0e7, "host": 1.0e7, "restart": 2.0e6, "adjoint": 1.2e7}[kind]
    while True:
        n = [int(round(math.exp(rng.uniform(math.log(14), math.log(200))))) for _ in range(3)]
        if rng.random() < 0.3:  # the sizes that people type
            n = [max(16, 8 * round(v / 8)) for v in n]
        ppc = round(math.exp(rng.uniform(math.log(3), math.log(64))), 2)
        total = 2 * ppc * n[0] * n[1] * n[2]
        if 1e5 <= total <= most and max(n) <= 8 * min(n):
            break
    steps = {"es": rng.randint(1, 12), "em": rng.randint(2, 16), "host": 1,
             "restart": rng.randint(1, 6), "adjoint": 2}[kind]
    ramp = rng.choice([0.0, 0.0, 20.0]) if kind == "es" else 0.0
    return dict(kind=kind, form=form, nx=n[0], ny=n[1], nz=n[2], ppc=ppc, steps=steps,
                wc=round(rng.uniform(0.0, 0.6), 3) if kind != "em" else 0.0, ramp=ramp)


# ---------------------------------------------------------------- parameters
def _grid(case):
    return case["nx"], case["ny"], case["nz"]


def _plasma(case):
    """Species (count, vth, drift), charges and units of a case, in the S-units
    of the reference (dt = 2, electron charge-to-mass ratio 1)."""
    n = _grid(case)
    vol = float(n[0] * n[1] * n[2])
    npin = int(round(case["ppc"] * vol))
    if case["kind"] == "em":  # background electrons and a 10% beam, ions at rest
        nb = int(round(0.1 * npin))
        dt, cv = 0.02, 20.0
        sp = [(-1.0, 1.0, npin, 1.0, 0.0), (-1.0, math.sqrt(0.1), nb, 1.0, 5.0)]
    elif case["kind"] == "adjoint":  # electrons and a 5% beam
        nb = int(round(0.05 * npin))
        dt, cv = 0.1, 0.0
        sp = [(-1.0, 1.0, npin, 1.0, 0.0), (-1.0, math.sqrt(0.05), nb, 1.0, 3.0)]
    else:  # electrons and ions of mass ratio 100
        dt, cv = (0.05 if case["ppc"] > 16 or case["ramp"] else 0.1), 0.0
        sp = [(-1.0, 1.0, npin, 1.0, 0.0), (0.01, 0.1, npin, 0.1, 0.0)]
    dth = dt / 2.0
    q_u = [wp * wp * vol / c / qm for qm, wp, c, _, _ in sp]
    q = [-v * dth * dth for v in q_u]
    qm = [-s[0] for s in sp]
    rm = [v / s[0] * dth * dth for v, s in zip(q_u, sp)]
    counts = [s[2] for s in sp]
    bk = -sum(a * b for a, b in zip(q, counts)) / vol
    return dict(n=n, counts=counts, vth=[s[3] * dth for s in sp], drift=[s[4] * dth for s in sp],
                q=q, qm=qm, rm=rm, b0=(0.0, 0.0, case["wc"] * dth), bk=bk, cs=(cv * dth) ** 2,
                ramp=case["ramp"])


def _device_species(p):
    return [dict(count=c, vth_perp=v, vth_para=v, drift=(d, 0.0, 0.0), ramp_ratio=p["ramp"])
            for c, v, d in zip(p["counts"], p["vth"], p["drift"])]


def _smooth_fields(p, seed):
    """A staggered eb(6, -1:n+1)^3 of a few long waves, as a host solver hands
    it over: [k, j, i, 6]."""
    r = np.random.RandomState(seed % (1 << 31))
    nx, ny, nz = p["n"]
    eb = np.zeros((nz + 3, ny + 3, nx + 3, 6))
    ax = [2.0 * np.pi * (np.arange(-1, m + 2) % m) / m for m in (nx, ny, nz)]
    for c in range(6):
        for _ in range(3):
            k = r.randint(1, 4, 3)
            ph = r.uniform(0.0, 2.0 * np.pi, 3)
            a = r.normal() * (2e-4 if c < 3 else 2e-3)
            eb[..., c] += (a * np.cos(k[2] * ax[2] + ph[2])[:, None, None]
                           * np.cos(k[1] * ax[1] + ph[1])[None, :, None]
                           * np.cos(k[0] * ax[0] + ph[0])[None, None, :])
    return eb


def _smooth_scalar(p, seed):
    return np.ascontiguousarray(1e3 * _smooth_fields(p, seed)[1:-2, 1:-2, 1:-2, 0])


def _records(p, seed):
    """The particle records of a snapshot: random order, numbered."""
    parts = []
    for s in range(len(p["counts"])):
        x, v = _particles(p, seed, s, 0, p["counts"][s])
        parts.append(torch.cat([x, v], dim=1))
    pv = torch.cat(parts).cpu().numpy()
    rec = np.zeros(len(pv), dtype=emg.PARTICLE)
    for c, name in enumerate(("x", "y", "z", "vx", "vy", "vz")):
        rec[name] = pv[:, c]
    rec["pid"] = np.arange(len(pv))
    rec["spec"] = np.repeat(np.arange(1, len(p["counts"]) + 1), p["counts"])
    return rec


# ----------------------------------------------------------------- the passes
def prepare(case, seed):
    p = _plasma(case)
    fp64 = case["form"] == "fp64"
    kind = case["kind"]
    kw = dict(precision=emg.PLAIN_FP64 if fp64 else emg.FP32_FIXED, b0=p["b0"])
    if kind == "restart" and not fp64:
        kw["track_pid"] = True
    if fp64 and kind not in ("adjoint", "restart"):
        kw["sort_every"] = 10
    ctx = emg.Context(p["n"], p["q"], p["qm"], p["rm"], p["counts"], **kw)
    st = dict(case=case, p=p, ctx=ctx)
    if kind == "restart":
        st["records"] = _records(p, seed)
        st["counts"] = np.array(p["counts"], dtype=np.int64)
    else:
        ctx.init_device(_device_species(p), seed)
    if kind in ("es", "em"):  # the initial field solve of a run
        ctx.deposit_rho(0)
        ctx.solve_es(p["bk"])
    else:
        st["eb"] = _smooth_fields(p, seed)
    if kind == "host":
        st["rho"] = np.zeros(tuple(m + 3 for m in reversed(p["n"])))
    if kind == "restart":
        ctx.set_fields(st["eb"])
    if kind == "adjoint":  # the states of a checkpoint window
        ctx.set_fields(st["eb"])
        for j in range(case["steps"]):
            ctx.state_save(j)
            ctx.push_es(2)
        ctx.state_save(case["steps"])
        st["g"] = [_smooth_scalar(p, seed + 17 + j) for j in range(case["steps"] + 1)]
    return st


def run(state):
    case, p, ctx = state["case"], state["p"], state["ctx"]
    kind, steps = case["kind"], case["steps"]
    if kind == "es":
        for _ in range(steps):
            ctx.push_es(2)
            ctx.deposit_rho(0)
            ctx.solve_es(p["bk"])
        return dict(rho=ctx.rho(), energy=ctx.energy(), field_energy=ctx.field_energy(p["cs"]))
    if kind == "em":
        for _ in range(steps):
            ctx.bfield()
            ctx.grdcrt()
            ctx.push_em(2)
            ctx.bfield()
            ctx.efield(2.0 * p["cs"], 2.0)
        return dict(eb=ctx.fields(), energy=ctx.energy(), field_energy=ctx.field_energy(p["cs"]))
    if kind == "host":
        ctx.set_fields(state["eb"])
        ctx.push_es(2)
        ctx.charge(0, rho=state["rho"])
        return dict(rho=state["rho"], energy=ctx.energy())
    if kind == "restart":
        ctx.upload(state["records"], state["counts"])
        for _ in range(steps):
            ctx.push_es(2)
        got, _ = ctx.download()
        rec = got.view(np.float64).reshape(-1, 8)
        if case["form"] == "fp32":  # whose tile buckets keep no order
            back = torch.empty(rec.shape, dtype=torch.float64)
            back[torch.from_numpy(got["pid"].astype(np.int64))] = torch.from_numpy(rec)
            rec = back.numpy()
        return {name: rec[:, c] for c, name in enumerate(("x", "y", "z", "vx", "vy", "vz"))}
    out = {}
    ctx.adj_reset()
    ctx.state_load(steps)
    ctx.adj_add_density(state["g"][steps], p["q"])
    for j in range(steps - 1, -1, -1):
        ctx.state_load(j)
        ctx.adj_step(2)
        out["field%d" % j] = ctx.adj_field()
        ctx.adj_add_density(state["g"][j], p["q"])
    out["velocity_sums"] = ctx.adj_velocity_sums()
    return out


def work(case):
    p = _plasma(case)
    n, total, ns = p["n"], float(sum(p["counts"])), len(p["counts"])
    ncell = float(n[0] * n[1] * n[2])
    nall = float((n[0] + 3) * (n[1] + 3) * (n[2] + 3))
    k, kind, steps = (96.0 if case["form"] == "fp64" else 56.0), case["kind"], case["steps"]
    w = 48.0 if case["form"] == "fp64" else 24.0
    if kind == "es":  # state in and out, nodes in, rho out; rho -> E -> nodes
        step = k * total + w * ncell + 8.0 * ns * ncell + (8.0 * ns + 24.0 + 24.0 + w) * ncell
        return dict(bytes=steps * step + 16.0 * ncell, flops=steps * 250.0 * total)
    if kind == "em":  # state, nodes, J; two B half steps, E, relocation
        step = k * total + w * ncell + 24.0 * ns * ncell + (72.0 + 24.0 * ns + 72.0 + 48.0 + w + 72.0) * ncell
        return dict(bytes=steps * step + 96.0 * nall, flops=steps * 450.0 * total)
    if kind == "host":  # eb in (host), relocation, step, rho out (host)
        return dict(bytes=(96.0 + 2 * w) * nall + k * total + 8.0 * ns * ncell + 16.0 * nall,
                    flops=250.0 * total)
    if kind == "restart":
        return dict(bytes=(64.0 + k / 2) * 2.0 * total + steps * (k * total + (w + 8.0 * ns) * ncell),
                    flops=steps * 250.0 * total)
    # state loaded, state and adjoints in, adjoints out, field out; density
    step = 96.0 * total + (24.0 + 96.0) * total + (48.0 + 24.0 + 24.0) * ncell \
        + (24.0 + 48.0) * total + 16.0 * ncell
    return dict(bytes=steps * step, flops=steps * 400.0 * total)


# ------------------------------------------------ the same in 64-bit torch
def _dev():
    return torch.device("cuda" if torch.cuda.is_available() else "cpu")


def _u01(seed, ctr):
    """The seeded counter-based stream of the device initialiser: SplitMix64
    over a counter, 53 bits, in (0, 1)."""
    def i64(v):
        v &= (1 << 64) - 1
        return v - (1 << 64) if v >= 1 << 63 else v

    def shr(z, s):
        return (z >> s) & ((1 << (64 - s)) - 1)

    z = ctr * i64(0x9E3779B97F4A7C15) + i64(seed)
    z = (z ^ shr(z, 30)) * i64(0xBF58476D1CE4E5B9)
    z = (z ^ shr(z, 27)) * i64(0x94D049BB133111EB)
    z = z ^ shr(z, 31)
    return (shr(z, 11).double() + 0.5) * (1.0 / 9007199254740992.0)


def _particles(p, seed, s, a, b):
    """Positions and velocities of particles a..b-1 of species s."""
    m = torch.arange(a, b, dtype=torch.int64, device=_dev())
    base = ((s << 40) + m) * 8
    u = [_u01(seed, base + k) for k in range(7)]
    n = p["n"]
    z = u[2]
    if p["ramp"] > 1.0:
        z = torch.log1p(z * (p["ramp"] - 1.0)) / math.log(p["ramp"])
    x = torch.stack([u[0] * n[0], u[1] * n[1], z * n[2]], dim=1)
    for d in range(3):
        x[:, d][x[:, d] >= n[d]] = 0.0
    r1, r2 = torch.sqrt(-2.0 * torch.log(u[3])), torch.sqrt(-2.0 * torch.log(u[5]))
    t1, t2 = 2.0 * math.pi * u[4], 2.0 * math.pi * u[6]
    v = p["vth"][s] * torch.stack([r1 * torch.cos(t1), r1 * torch.sin(t1), r2 * torch.cos(t2)], dim=1)
    v[:, 0] += p["drift"][s]
    return x, v


def _corners(x, n):
    """Cell (as float) and, corner by corner, the periodic node index and the
    trilinear weight."""
    c = torch.floor(x)
    i = c.long()
    f = x - c
    for q in range(8):
        idx, w = None, None
        for d in (2, 1, 0):
            o = (q >> d) & 1
            g = (i[:, d] + o) % n[d]
            idx = g if idx is None else idx * n[d] + g
            wd = f[:, d] if o else 1.0 - f[:, d]
            w = wd if w is None else w * wd
        yield idx, w


def _nodes(e, b, b0):
    """Relocation of the staggered E, B [nz, ny, nx, 3] to the nodes, [ncell, 6]."""
    def back(a, d):
        return torch.roll(a, 1, 2 - d)

    out = [0.5 * (e[..., d] + back(e[..., d], d)) for d in range(3)]
    for d in range(3):
        u, w = [a for a in range(3) if a != d]
        c = b[..., d]
        out.append(0.25 * (c + back(c, u) + back(c, w) + back(back(c, u), w)) + b0[d])
    return torch.stack(out, dim=-1).reshape(-1, 6)


def _rotate(v, t):
    """Buneman-Boris rotation by the half-step vector t."""
    s = 2.0 / (1.0 + (t * t).sum(1, keepdim=True))
    vp = v + torch.linalg.cross(v, t)
    return v + s * torch.linalg.cross(vp, t)


def _push(x, v, node, n, qmp):
    f = None
    for idx, w in _corners(x, n):
        t = node[idx] * w[:, None]
        f = t if f is None else f.add_(t)
    v = v + qmp * f[:, :3]
    v = _rotate(v, qmp * f[:, 3:])
    return v + qmp * f[:, :3]


def _wrap(x, n):
    box = torch.tensor([float(m) for m in n], dtype=torch.float64, device=x.device)
    x = torch.where(x < 0.0, x + box, x)
    return torch.where(x >= box, x - box, x)


def _chunks(xs):
    for s, x in enumerate(xs):
        for a in range(0, len(x), CHUNK):
            yield s, slice(a, min(a + CHUNK, len(x)))


def _deposit(xs, n, q):
    rho = torch.zeros(n[0] * n[1] * n[2], dtype=torch.float64, device=_dev())
    for s, c in _chunks(xs):
        for idx, w in _corners(xs[s][c], n):
            rho.index_add_(0, idx, w, alpha=q[s])
    return rho.reshape(n[2], n[1], n[0])


def _solve(rho):
    """E = -grad phi of the 7-point periodic Poisson equation."""
    def eig(m):
        return (2.0 * torch.sin(math.pi * torch.arange(m, dtype=torch.float64, device=rho.device) / m)) ** 2

    nz, ny, nx = rho.shape
    div = eig(nz)[:, None, None] + eig(ny)[None, :, None] + eig(nx)[None, None, :]
    div[0, 0, 0] = 1.0
    spec = torch.fft.fftn(rho) / div
    spec[0, 0, 0] = 0.0
    phi = torch.fft.ifftn(spec).real
    return torch.stack([phi - torch.roll(phi, -1, 2 - d) for d in range(3)], dim=-1)


def _move(xs, vs, node, p):
    n = p["n"]
    for s, c in _chunks(xs):
        vs[s][c] = _push(xs[s][c], vs[s][c], node, n, p["qm"][s])
        xs[s][c] = _wrap(xs[s][c] + 2.0 * vs[s][c], n)


def _segment(j, r0, r1, cell, n, q):
    """One zigzag segment r0 -> r1 in the cell `cell` (as float)."""
    i = cell.long()
    flux = (r1 - r0) * (0.5 * q)
    m = 0.5 * (r0 + r1) - cell
    for d in range(3):
        u, w = [a for a in range(3) if a != d]
        for ou in (0, 1):
            for ow in (0, 1):
                g = [i[:, 0], i[:, 1], i[:, 2]]
                g[u] = g[u] + ou
                g[w] = g[w] + ow
                idx = ((g[2] % n[2]) * n[1] + g[1] % n[1]) * n[0] + g[0] % n[0]
                wt = (m[:, u] if ou else 1.0 - m[:, u]) * (m[:, w] if ow else 1.0 - m[:, w])
                j[d].index_add_(0, idx, flux[:, d] * wt)


def _zigzag(xs, vs, node, p):
    """Push, move, and the zigzag current [nz, ny, nx, 3]."""
    n = p["n"]
    dev = _dev()
    j = torch.zeros((3, n[0] * n[1] * n[2]), dtype=torch.float64, device=dev)
    box = torch.tensor([float(m) for m in n], dtype=torch.float64, device=dev)
    for s, c in _chunks(xs):
        x0 = xs[s][c].clone()
        vs[s][c] = _push(x0, vs[s][c], node, n, p["qm"][s])
        x1 = x0 + 2.0 * vs[s][c]
        ca, cb = torch.floor(x0), torch.floor(x1)
        low, high = x1 < 0.0, x1 >= box  # through a face of the box: relay on that face
        cb = torch.where(low, torch.full_like(cb, -1.0), torch.where(high, box.expand_as(cb), cb))
        r = torch.where(ca == cb, 0.5 * (x0 + x1), torch.maximum(ca, cb))
        _segment(j, x0, r, ca, n, p["q"][s])
        _segment(j, r, x1, cb, n, p["q"][s])
        xs[s][c] = _wrap(x1, n)
    return j.reshape(3, n[2], n[1], n[0]).permute(1, 2, 3, 0)


def _b_half(e, b):
    def up(a, d):
        return torch.roll(a, -1, 2 - d)

    return torch.stack([b[..., d] + (up(e[..., (d + 1) % 3], (d + 2) % 3) - e[..., (d + 1) % 3])
                        - (up(e[..., (d + 2) % 3], (d + 1) % 3) - e[..., (d + 2) % 3])
                        for d in range(3)], dim=-1)


def _e_full(e, b, aj, tcs):
    def dn(a, d):
        return torch.roll(a, 1, 2 - d)

    return torch.stack([e[..., d] + tcs * ((b[..., (d + 2) % 3] - dn(b[..., (d + 2) % 3], (d + 1) % 3))
                                           - (b[..., (d + 1) % 3] - dn(b[..., (d + 1) % 3], (d + 2) % 3)))
                        - 2.0 * aj[..., d] for d in range(3)], dim=-1)


def _kinetic(vs, p):
    vol = float(p["n"][0] * p["n"][1] * p["n"][2])
    out = [[0.5 * p["rm"][s] * float(sum((vs[s][a:a + CHUNK, d] ** 2).sum()
                                         for a in range(0, len(vs[s]), CHUNK))) / vol
            for d in range(3)] for s in range(len(vs))]
    return np.array(out)


def _field_energy(e, b, cs):
    vol = float(e[..., 0].numel())
    return np.array([0.5 * float((e * e).sum()) / vol, 0.5 * cs * float((b * b).sum()) / vol])


def _halo(e, b):
    eb = torch.cat([e, b], dim=-1)
    for d in range(3):
        m = eb.shape[d]
        at = (torch.arange(-1, m + 2, device=eb.device)) % m
        eb = eb.index_select(d, at)
    return eb


def _ghosted_rho(xs, p):
    """rho(-1:n+1)^3 as the border exchange and the boundary fold leave it: the
    nodes 0..n hold the periodic sum, ghost -1 the raw deposit of node n and
    ghost n + 1 that of node 0, folded along z for a y ghost inside z 0..n and
    along y and z for an x ghost inside y, z 0..n."""
    n = p["n"]
    m = [v + 1 for v in n]
    raw = torch.zeros(m[0] * m[1] * m[2], dtype=torch.float64, device=_dev())
    for s, c in _chunks(xs):
        for idx, w in _corners(xs[s][c], [v + 2 for v in n]):  # no node is beyond n
            i = idx % (n[0] + 2)
            j = idx // (n[0] + 2) % (n[1] + 2)
            k = idx // ((n[0] + 2) * (n[1] + 2))
            raw.index_add_(0, (k * m[1] + j) * m[0] + i, w, alpha=p["q"][s])
    raw = raw.reshape(m[2], m[1], m[0]).cpu().numpy()

    def sets(t, v, fold):
        if t == -1:
            return [v]
        if t == v + 1:
            return [0]
        return [0, v] if fold and t in (0, v) else [t]

    def axis(a, ax, v, fold):
        rows = [a.take(sets(t, v, fold), axis=ax).sum(axis=ax) for t in range(-1, v + 2)]
        return np.stack(rows, axis=ax)

    z = axis(raw, 0, n[2], True)
    out = np.empty((n[2] + 3, n[1] + 3, n[0] + 3))
    kin = slice(1, n[2] + 2)
    y = axis(z, 1, n[1], False)
    y[kin] = axis(z[kin], 1, n[1], True)
    out[...] = axis(y, 2, n[0], False)
    jin = slice(1, n[1] + 2)
    out[kin, jin] = axis(y[kin, jin], 2, n[0], True)
    return out


def _compact(eb, p):
    n = p["n"]
    t = torch.from_numpy(eb).to(_dev())[1:1 + n[2], 1:1 + n[1], 1:1 + n[0]]
    return t[..., :3], t[..., 3:]


def _adjoint_step(x, lx, lv, node, n, qmp, acc):
    """Reverse of one push at position x: the adjoints before it, the adjoint
    of the nodal E added to acc [ncell, 3]."""
    f, bf = [], None
    for idx, w in _corners(x, n):
        t = node[idx]
        f.append(t[:, :3])
        bf = w[:, None] * t[:, 3:] if bf is None else bf + w[:, None] * t[:, 3:]
    w3 = lv + 2.0 * lx
    mt = _rotate(w3, -qmp * bf)
    la = mt + w3
    lx = lx + qmp * _gradient(x, [(la * e).sum(1) for e in f], n)
    for idx, w in _corners(x, n):
        acc.index_add_(0, idx, (qmp * w)[:, None] * la)
    return lx, mt


def _gradient(x, s, n):
    """Gradient of the trilinear interpolant of the corner values s."""
    f = x - torch.floor(x)
    out = torch.zeros_like(x)
    for q in range(8):
        o = [(q >> d) & 1 for d in range(3)]
        wd = [f[:, d] if o[d] else 1.0 - f[:, d] for d in range(3)]
        for d in range(3):
            u, w = [a for a in range(3) if a != d]
            out[:, d] += s[q] * (1.0 if o[d] else -1.0) * wd[u] * wd[w]
    return out


def exact(case, seed):
    p = _plasma(case)
    n, kind, steps = p["n"], case["kind"], case["steps"]
    xs = [torch.empty((c, 3), dtype=torch.float64, device=_dev()) for c in p["counts"]]
    vs = [torch.empty_like(x) for x in xs]
    for s, c in _chunks(xs):
        xs[s][c], vs[s][c] = _particles(p, seed, s, c.start, c.stop)
    if kind in ("es", "em"):
        rho = _deposit(xs, n, p["q"])
        e = _solve(rho + p["bk"])
        b = torch.zeros_like(e)
    else:
        e, b = _compact(_smooth_fields(p, seed), p)
    if kind == "es":
        for _ in range(steps):
            _move(xs, vs, _nodes(e, b, p["b0"]), p)
            rho = _deposit(xs, n, p["q"])
            e = _solve(rho + p["bk"])
        return dict(rho=rho, energy=_kinetic(vs, p), field_energy=_field_energy(e, b, p["cs"]))
    if kind == "em":
        for _ in range(steps):
            b = _b_half(e, b)
            aj = _zigzag(xs, vs, _nodes(e, b, p["b0"]), p)
            b = _b_half(e, b)
            e = _e_full(e, b, aj, 2.0 * p["cs"])
        return dict(eb=_halo(e, b), energy=_kinetic(vs, p),
                    field_energy=_field_energy(e, b, p["cs"]))
    node = _nodes(e, b, p["b0"])
    if kind == "host":
        _move(xs, vs, node, p)
        return dict(rho=_ghosted_rho(xs, p), energy=_kinetic(vs, p))
    if kind == "restart":
        for _ in range(steps):
            _move(xs, vs, node, p)
        x, v = torch.cat(xs), torch.cat(vs)
        return dict(x=x[:, 0], y=x[:, 1], z=x[:, 2], vx=v[:, 0], vy=v[:, 1], vz=v[:, 2])
    states = []
    for _ in range(steps):
        states.append([x.clone() for x in xs])
        _move(xs, vs, node, p)
    states.append(xs)
    g = [torch.from_numpy(_smooth_scalar(p, seed + 17 + j)).to(_dev()).reshape(-1)
         for j in range(steps + 1)]

    def density(x, gj, q):
        return q * _gradient(x, [gj[idx] for idx, _ in _corners(x, n)], n)

    lx = [density(x, g[steps], q) for x, q in zip(states[steps], p["q"])]
    lv = [torch.zeros_like(x) for x in lx]
    out = {}
    for j in range(steps - 1, -1, -1):
        acc = torch.zeros((n[0] * n[1] * n[2], 3), dtype=torch.float64, device=_dev())
        for s, x in enumerate(states[j]):
            lx[s], lv[s] = _adjoint_step(x, lx[s], lv[s], node, n, p["qm"][s], acc)
            lx[s] = lx[s] + density(x, g[j], p["q"][s])
        out["field%d" % j] = acc.reshape(n[2], n[1], n[0], 3)
    out["velocity_sums"] = torch.stack([v.sum(0) for v in lv])
    return out
