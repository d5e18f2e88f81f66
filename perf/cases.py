"""The work that programs have this package do, as cases that can be timed.

Four kinds of case, each through the public entry points:

* "run": one periodic box from one dump to the next.  A program steps the box
  `steps` times (in calls of `per_call` steps: 1 is the Fortran driver's loop,
  which prints the CFL number of every step; 0 is one call for all of them)
  and then copies the fields out, as it does at every dump.  The state goes on
  from pass to pass, as a run does.
* "batch": up to 16 boxes stepped together by step_batch, then copied out.
* "serve": an Ensemble that takes a set of requests (parameters and initial
  fields in host memory), steps them to their ends and gives their fields back.
* "drops": the post-processing of one dump on the device: the drop list
  (count, volumes, equivalent diameters) and the energy diagnostics.

Initial fields are random-phase solenoidal velocity with the spectrum
k^4 exp(-2 (k/k_p)^2), u_rms = 1, and spherical drops of tanh profile on a
jittered lattice.  The ABC forcing is held against the viscosity at the
laminar amplitude `force`, dt is 0.02 dx, and the viscosity follows the
resolution, so that a run stays bounded however long it is continued.
"""
import math
import random

import numpy as np
import torch

FIELD = {"u": 1, "v": 2, "w": 3, "p": 4, "phi": 5}
SIZES = sorted(2 ** a * 3 ** b for a in range(1, 10) for b in range(0, 6) if 16 <= 2 ** a * 3 ** b <= 512)


def _case(name, kind="run", nx=128, precision="fp64", phi=True, steps=100, per_call=0, drops=2, force=0.5,
          wavenumbers="reference", rhs="fp32", sizes="", requests=0):
    """`drops`: drops per direction of the lattice.  `sizes`: the boxes' nx for
    "batch" and "serve", by commas."""
    return dict(name=name, kind=kind, nx=nx, precision=precision, phi=phi, steps=steps, per_call=per_call,
                drops=drops, force=force, wavenumbers=wavenumbers, rhs=rhs, sizes=sizes, requests=requests)


def listed():
    return [
        # the smallest box of the test suite under the Fortran driver's loop: one call per step,
        # so launches and the wait at the end of each call are all there is
        _case("driver_32", nx=32, steps=200, per_call=1, drops=1),
        # a small FP64 box advanced from dump to dump in one call
        _case("box_64", nx=64, steps=1000, drops=2),
        # a serving-size box in mixed precision whose length has a factor 3
        _case("box_96_mixed", nx=96, precision="mixed", steps=600, drops=2),
        # a ragged length (4 * 27) that no tile divides, single phase, unforced decay
        _case("decay_108", nx=108, phi=False, steps=500, force=0.0),
        # the reference's default size, single phase, under the driver's loop (its validation run)
        _case("driver_128", nx=128, phi=False, steps=500, per_call=1),
        # the larger serving size in mixed precision, factor 3
        _case("box_192_mixed", nx=192, precision="mixed", steps=400, drops=3),
        # forced turbulence with 64 drops, FP64, and the projection that is exact to round-off
        # (finite-difference wavenumbers, right-hand side not rounded)
        _case("hit_256", nx=256, steps=250, drops=4, wavenumbers="modified", rhs="fp64"),
        # the headline workload, 512^3 with 512 drops in FP64, between two dumps
        _case("hit_512", nx=512, steps=120, drops=8),
        # the same box in mixed precision
        _case("hit_512_mixed", nx=512, precision="mixed", steps=100, drops=8),
        # eight small boxes of a parameter study stepped together
        _case("batch_64", kind="batch", precision="mixed", steps=300, sizes="64,64,64,64,64,64,64,64"),
        # a serving process answering a burst of uneven requests, mixed precision
        _case("serve_burst", kind="serve", precision="mixed", steps=200, requests=10,
              sizes="64,96,64,128,64,96,64,64,128,64"),
        # drop statistics and energies of a 256^3 dump with 64 drops
        _case("drops_256", kind="drops", nx=256, drops=4, steps=0),
    ]


def draw(rng):
    def size(lo, hi):
        x = math.exp(rng.uniform(math.log(lo), math.log(hi)))
        return min((s for s in SIZES if lo <= s <= hi), key=lambda s: abs(math.log(s / x)))

    precision = rng.choice(["fp64", "mixed"])
    force = rng.choice([0.0, 0.25, 0.5])
    kind = rng.choice(["run"] * 7 + ["batch", "serve", "drops", "drops"])
    if kind == "batch":
        sizes = sorted(size(16, 128) for _ in range(rng.randint(2, 8)))
        return _case("", kind, sizes=",".join(map(str, sizes)), precision=precision, steps=rng.randint(50, 300),
                     phi=rng.random() < 0.6, force=force)
    if kind == "serve":
        k = rng.randint(3, 10)
        return _case("", kind, sizes=",".join(str(size(32, 128)) for _ in range(k)), requests=k, precision=precision,
                     steps=rng.randint(50, 300), force=force)
    n = size(16, 512)
    lattice = rng.randint(1, max(1, n // 40))
    if kind == "drops":
        return _case("", kind, nx=n, drops=lattice, precision=precision, steps=0)
    most = int(min(1000, 100 * (512 / n) ** 3))
    return _case("", kind, nx=n, precision=precision, phi=rng.random() < 0.6, steps=rng.randint(max(1, most // 4), most),
                 per_call=rng.choice([0, 0, 1, 10]), drops=lattice, force=force,
                 wavenumbers=rng.choice(["reference", "reference", "modified"]), rhs=rng.choice(["fp32", "fp32", "fp64"]))


# -- inputs ---------------------------------------------------------------------

def _device():
    return torch.device("cuda" if torch.cuda.is_available() else "cpu")


def _grid(n):
    dx = 2.0 * math.pi / (n - 1)
    return dx, torch.arange(n, dtype=torch.float64, device=_device()) * dx


def _velocity(n, seed):
    """u, v, w as [z, y, x] tensors: the staggered curl of a random-phase potential."""
    dev, dx = _device(), _grid(n)[0]
    g = torch.Generator(device=dev).manual_seed(seed)
    k1 = torch.fft.fftfreq(n, 1.0 / n, dtype=torch.float64, device=dev)
    kr = torch.arange(n // 2 + 1, dtype=torch.float64, device=dev)
    k2 = k1[:, None, None] ** 2 + k1[None, :, None] ** 2 + kr[None, None, :] ** 2
    kp = min(4.0, n / 8.0)
    amp = torch.where((k2 > 0) & (k2 <= min(n // 2 - 1, 6 * kp) ** 2), torch.exp(-k2 / kp ** 2), torch.zeros_like(k2))
    a = []
    for _ in range(3):
        z = torch.randn((2,) + tuple(k2.shape), dtype=torch.float64, device=dev, generator=g)
        a.append(torch.fft.irfftn(torch.complex(z[0], z[1]) * amp, s=(n, n, n)))
    ax, ay, az = a

    def d(f, axis):
        return (torch.roll(f, -1, axis) - f) / dx

    u, v, w = d(az, 1) - d(ay, 0), d(ax, 0) - d(az, 2), d(ay, 2) - d(ax, 1)
    s = 1.0 / math.sqrt(float(((u * u).mean() + (v * v).mean() + (w * w).mean()) / 3.0))
    return [u * s, v * s, w * s]


def _drops(n, per_side, seed):
    """Drops of radius ~0.28 lattice spacings, jittered, on a per_side^3 lattice: [z, y, x]."""
    dx, x = _grid(n)
    dev = x.device
    r = np.random.default_rng(seed)
    period = n * dx
    cell = period / per_side
    phi = torch.zeros((n, n, n), dtype=torch.float64, device=dev)
    for q in range(per_side ** 3):
        c = (np.array([q % per_side, (q // per_side) % per_side, q // per_side ** 2]) + 0.5) * cell
        c = c + r.uniform(-0.08, 0.08, 3) * cell
        radius = float(r.uniform(0.24, 0.32)) * cell
        half = int((radius + 40.0 * dx) / dx) + 2
        span = (-half, half + 1) if 2 * half + 1 <= n else (-(n // 2), n - n // 2)
        at, dist = [], []
        for m in range(3):
            i = torch.arange(*span, device=dev) + int(round(c[m] / dx))
            dist.append((i.to(torch.float64) * dx - float(c[m])) ** 2)
            at.append(i % n)
        rr = torch.sqrt(dist[2][:, None, None] + dist[1][None, :, None] + dist[0][None, None, :])
        box = (at[2][:, None, None], at[1][None, :, None], at[0][None, None, :])
        phi[box] = torch.maximum(phi[box], 0.5 * (1.0 - torch.tanh((rr - radius) / 2.0 / dx)))
    return phi


def _boxes(case, seed):
    """The boxes of a case: (parameters by name, steps, {field: [z, y, x] tensor})."""
    if case["kind"] in ("batch", "serve"):
        sizes = [int(s) for s in case["sizes"].split(",")]
    else:
        sizes = [case["nx"]]
    r = random.Random(seed)
    out = []
    for b, n in enumerate(sizes):
        phi = bool(case["phi"]) if case["kind"] != "serve" else b % 2 == 0
        lattice = case["drops"] if len(sizes) == 1 else max(1, n // 48)
        dx = 2.0 * math.pi / (n - 1)
        mu = 0.006 * 128 / n * (1.0 if len(sizes) == 1 else r.uniform(0.8, 1.5))
        steps = case["steps"] if case["kind"] != "serve" else r.randint(case["steps"] // 2, case["steps"])
        f = case["force"] * mu * 4.0
        p = dict(nx=n, dt=0.02 * dx, mu=mu, rho=1.0, f1=f, f2=f, f3=f, k0=2.0, radius=0.5, sigma=0.05, epsr=1.0,
                 gamma_factor=1.2, phiflag=int(phi), inflow=1, inphi=int(phi),
                 precision=int(case["precision"] == "mixed"), wavenumbers=int(case["wavenumbers"] == "modified"),
                 poisson_rhs_fp32=int(case["rhs"] == "fp32"))
        fields = dict(zip("uvw", _velocity(n, seed * 64 + b)))
        if phi:
            fields["phi"] = _drops(n, lattice, seed * 64 + b)
        out.append((p, steps, fields))
    return out


def _host(t):
    """A [z, y, x] tensor as the package's [x, y, z] array of Fortran order."""
    return t.cpu().numpy().transpose(2, 1, 0)


# -- the package -------------------------------------------------------------------

def prepare(case, seed):
    import mhit36_amd

    state = {"kind": case["kind"], "steps": case["steps"], "per_call": case["per_call"] or case["steps"]}
    boxes = _boxes(case, seed)
    if case["kind"] == "serve":
        state["server"] = mhit36_amd.Ensemble(hbm_budget_bytes=4 << 30, autotune=False)
        state["requests"] = [(p, steps, {k: _host(t) for k, t in fields.items()}) for p, steps, fields in boxes]
        return state
    state["boxes"] = []
    for p, _, fields in boxes:
        s = mhit36_amd.Solver(**p)
        for name, t in fields.items():
            s.set_field(FIELD[name], _host(t))
        state["boxes"].append(s)
    return state


def _fields(box):
    return {name: box.get_field(k) for name, k in FIELD.items() if name != "phi" or box.params.phiflag}


def run(state):
    import mhit36_amd

    if state["kind"] == "run":
        box = state["boxes"][0]
        left = state["steps"]
        while left > 0:
            d = box.step(min(left, state["per_call"]))
            left -= state["per_call"]
        return {"umax": d.gumax, "cfl": d.cou, **_fields(box)}
    if state["kind"] == "batch":
        d = mhit36_amd.solver.step_batch(state["boxes"], state["steps"])
        return [{"umax": x.gumax, **_fields(s)} for x, s in zip(d, state["boxes"])]
    if state["kind"] == "drops":
        box = state["boxes"][0]
        count, volume, deq = box.drop_count()
        return {"count": count, "volume": volume, "deq": deq, **box.diagnostics()}
    server, out = state["server"], []
    ids = [server.submit(dict(p), nsteps=steps, **fields) for p, steps, fields in state["requests"]]
    server.wait_idle()
    server.results()
    for rid, (p, _, _) in zip(ids, state["requests"]):
        out.append({name: server.get_field(rid, k) for name, k in FIELD.items() if name != "phi" or p["phiflag"]})
        server.release(rid)
    return out


def work(case):
    """A step reads and writes the velocity, the previous right-hand side and
    phi once (14 values per cell, 12 without phi), and the transform moves the
    half spectrum through memory once each way (2 values); a dump reads the
    fields.  Arithmetic: the two transforms, and the stencils."""
    total_b = total_f = 0.0
    boxes = [(case["nx"], case["phi"])]
    if case["kind"] in ("batch", "serve"):
        boxes = [(int(n), case["phi"] if case["kind"] == "batch" else b % 2 == 0)
                 for b, n in enumerate(case["sizes"].split(","))]
    width = 4.0 if case["precision"] == "mixed" else 8.0
    for n, phi in boxes:
        cells = float(n) ** 3
        fields = 4 if not phi else 5
        if case["kind"] == "drops":
            total_b += cells * 4 * width
            total_f += cells * 60.0
            continue
        steps = case["steps"] * (0.75 if case["kind"] == "serve" else 1.0)
        total_b += cells * (steps * ((14 if phi else 12) * width + 32.0) + fields * 8.0)
        total_f += cells * steps * (5.0 * math.log2(cells) + (400.0 if phi else 150.0))
    return {"bytes": total_b, "flops": total_f}


# -- the same in plain torch, 64 bits -------------------------------------------------

def _steps64(p, steps, fields):
    """`steps` steps of one fresh box (the first is an Euler step), as the
    equations are discretised in multi/main.f90:338-946: the fields at the end."""
    n = p["nx"]
    dx, x = _grid(n)
    dxi, ddxi, dt, mu, rhoi = 1.0 / dx, 1.0 / dx / dx, p["dt"], p["mu"], 1.0 / p["rho"]
    eps, tiny = p["epsr"] * dx, float(np.float32(1.0e-16))
    X, Y, Z = 2, 1, 0

    def at(f, axis, by):                       # f at the neighbour `by` cells along `axis`
        return torch.roll(f, -by, axis)

    def central(f, axis):
        return (at(f, axis, 1) - at(f, axis, -1)) * (0.5 * dxi)

    def lap(f):
        return (at(f, X, 1) + at(f, X, -1) + at(f, Y, 1) + at(f, Y, -1) + at(f, Z, 1) + at(f, Z, -1) - 6.0 * f) * ddxi

    def flux(a, b):                            # face product of two averaged velocities
        return 0.25 * a * b

    k = torch.arange(n, dtype=torch.float64, device=x.device)
    k = torch.where(k < n // 2, k, k - n)
    if p["wavenumbers"]:
        k = 2.0 * dxi * torch.sin(math.pi * torch.arange(n, dtype=torch.float64, device=x.device) / n)
    k2 = k[:, None, None] ** 2 + k[None, :, None] ** 2 + k[None, None, :n // 2 + 1] ** 2
    k2[0, 0, 0] = 1.0
    sin, cos = torch.sin(p["k0"] * x), torch.cos(p["k0"] * x)
    force = (p["f3"] * sin[:, None, None] + p["f2"] * cos[None, :, None],
             p["f1"] * sin[None, None, :] + p["f3"] * cos[:, None, None],
             p["f2"] * sin[None, :, None] + p["f1"] * cos[None, None, :])
    u, v, w = fields["u"], fields["v"], fields["w"]
    phi, old, umax, pr = fields.get("phi"), None, 1.0, None
    for _ in range(steps):
        if phi is not None:
            f = torch.clamp(phi, max=1.0)
            a, b = f + tiny, (1.0 - f) + tiny
            psi = eps * torch.log(a / b)
            gx, gy, gz = (at(psi, m, 1) - at(psi, m, -1) for m in (X, Y, Z))
            s = a * b / (a + b) ** 2 / (torch.sqrt(gx * gx + gy * gy + gz * gz) + tiny)
            div = central(s * gx, X) + central(s * gy, Y) + central(s * gz, Z)
            r = 0.0
            for vel, m in ((u, X), (v, Y), (w, Z)):
                face = vel * 0.5 * (phi + at(phi, m, -1))
                r = r - (at(face, m, 1) - face) * dxi
            gamma = p["gamma_factor"] * umax
            phi = phi + dt * (r + gamma * (eps * lap(phi) - div))
        rhs = []
        for vel, axis in ((u, X), (v, Y), (w, Z)):
            r = mu * rhoi * lap(vel)
            for adv, m in ((u, X), (v, Y), (w, Z)):
                if m == axis:
                    c = flux(vel + at(vel, m, -1), vel + at(vel, m, -1))
                    r = r - (at(c, m, 1) - c) * dxi
                else:
                    c = flux(vel + at(vel, m, -1), adv + at(adv, axis, -1))
                    r = r - (at(c, m, 1) - c) * dxi
            rhs.append(r)
        rhs = [r + f for r, f in zip(rhs, force)]
        if phi is not None:
            chem = 6.0 * p["sigma"] * (phi * (1.0 - phi) * (1.0 - 2.0 * phi) / eps - eps * lap(phi))
            for q, m in enumerate((X, Y, Z)):
                c = chem * central(phi, m)
                rhs[q] = rhs[q] + 0.5 * (at(c, m, -1) + c) * rhoi
        old = rhs if old is None else old
        u, v, w = (f + dt * (1.5 * r - 0.5 * o) for f, r, o in zip((u, v, w), rhs, old))
        old = rhs
        q = (p["rho"] * dxi / dt) * ((at(u, X, 1) - u) + (at(v, Y, 1) - v) + (at(w, Z, 1) - w))
        if p["poisson_rhs_fp32"]:
            q = q.to(torch.float32).to(torch.float64)
        z = torch.fft.rfftn(q) / -k2
        z[0, 0, 0] = 0.0
        pr = torch.fft.irfftn(z, s=(n, n, n))
        new = []
        for f, m in ((u, X), (v, Y), (w, Z)):
            f = f - dt * rhoi * dxi * (pr - at(pr, m, -1))
            new.append(f - f.mean())
        u, v, w = new
        umax = float(max(u.max(), v.max(), w.max()))
    out = {"u": u, "v": v, "w": w, "p": pr}
    if phi is not None:
        out["phi"] = phi
    return out, umax


def _labels64(inside):
    """Each cell of a drop (26-connected, periodic) labelled by the smallest
    linear index of its drop, x fastest; others by the cell count."""
    n = inside.shape[0]
    none = n ** 3
    lab = torch.where(inside, torch.arange(none, device=inside.device).reshape(n, n, n), none)
    while True:
        low = lab
        for m in range(3):
            low = torch.minimum(low, torch.minimum(torch.roll(low, 1, m), torch.roll(low, -1, m)))
        low = torch.where(inside, low, none)
        if torch.equal(low, lab):
            return lab
        lab = low


def exact(case, seed):
    boxes = _boxes(case, seed)
    if sum(p["nx"] ** 3 * steps for p, steps, _ in boxes) > 1.7e10:
        return None                            # over 20 seconds
    if case["kind"] == "drops":
        p, _, f = boxes[0]
        n, dx = p["nx"], _grid(p["nx"])[0]
        stored = {k: (t.to(torch.float32).to(torch.float64) if p["precision"] else t) for k, t in f.items()}
        _, cells = torch.unique(_labels64(stored["phi"] >= 0.5)[stored["phi"] >= 0.5], return_counts=True)
        cells = cells.to(torch.float64).cpu()
        grad = [[(torch.roll(f[c], -1, m) - torch.roll(f[c], 1, m)) / (2.0 * dx) for m in (2, 1, 0)] for c in "uvw"]
        strain = sum(((grad[a][b] + grad[b][a]) / 2.0).square().mean() for a in range(3) for b in range(3))
        total = float(stored["phi"].sum())
        return {"count": None, "volume": cells, "deq": dx * (6.0 * cells / math.pi) ** (1.0 / 3.0),
                "ke": 0.5 * float(sum(f[c].square().mean() for c in "uvw")),
                "diss": 2.0 * p["mu"] / p["rho"] * float(strain), "phi_sum": total, "phi_volume": total * dx ** 3}
    out = []
    for p, steps, fields in boxes:
        end, umax = _steps64(p, steps, fields)
        end = {k: t.permute(2, 1, 0).cpu() for k, t in end.items()}
        if case["kind"] == "run":
            end = {"umax": umax, "cfl": umax * p["dt"] * (p["nx"] - 1) / (2.0 * math.pi), **end}
        elif case["kind"] == "batch":
            end = {"umax": umax, **end}
        out.append(end)
    return out[0] if case["kind"] == "run" else out
