"""What this framework is used for, as cases whose time can be measured.

A case is a program that holds a machine (or a batch of them), advances it by an output
interval of time steps and reads the fields out, or differentiates a rollout.  ``run`` is one
such interval through the public entry points; the state goes on from where the last interval
left it, as in a simulation.  ``exact`` computes the first interval in 64 bits with torch alone.
"""
import math

import numpy as np
import torch

from paraiso_amd import inputs, variants
from paraiso_amd.autograd import rollout

HYDRO = ("density", "velocity0", "velocity1", "pressure")
GAMMA = 1.4
# operations of a cell update as the schemes write them (each value once per cell)
OPS = {"hydro": 777, "life": 12, "wave": 16}


def listed():
    return [
        # the headline program, a Kelvin-Helmholtz run at full size: the carried-CFL step
        # replayed as a HIP graph between two outputs
        dict(name="hydro_f32_2048", kind="hydro", variant="hydro_f32", nx=2048, ny=2048,
             kernel="proceed_pipelined", steps=20, graph=True),
        # the reference's own step (CFL pass, then update) on a ragged mid-size grid, call by call
        dict(name="hydro_f32_ragged", kind="hydro", variant="hydro_f32", nx=1021, ny=767,
             kernel="proceed", steps=10, graph=False),
        # a quick look at a small grid: launches and latency
        dict(name="hydro_f32_small", kind="hydro", variant="hydro_f32", nx=96, ny=64,
             kernel="proceed", steps=16, graph=False),
        # the double precision run that single precision is checked against
        dict(name="hydro_f64_1024", kind="hydro", variant="hydro_f64", nx=1024, ny=1024,
             kernel="proceed_pipelined", steps=10, graph=True),
        # a parameter study: 256 grids of uneven sizes advanced together
        dict(name="hydro_batch_256", kind="batch", variant="hydro_f32_batch", grids=256,
             lo=64, hi=1024, kernel="proceed_pipelined", steps=40, graph=True),
        # gradient of the kinetic energy in a square after a rollout, forward and backward
        dict(name="hydro_grad_512", kind="hydro_grad", variant="hydro_adj2_f32_fast", nx=512,
             ny=512, steps=40, every=20),
        # Life at its benchmark size: 1000 generations, eight per launch, one graph
        dict(name="life_1024_x8", kind="life", variant="life_i32", nx=1024, ny=1024,
             kernel="proceed_x8", per=8, steps=125, graph=True),
        # Life as the reference calls it, generation by generation, on an odd grid
        dict(name="life_odd", kind="life", variant="life_i32", nx=333, ny=217,
             kernel="proceed", per=1, steps=100, graph=False),
        # the 3-D wave at its benchmark size, two steps per launch
        dict(name="wave_512_x2", kind="wave", variant="wave3d_f32", nx=512, ny=512, nz=512,
             kernel="proceed_x2", per=2, steps=20, graph=False),
        # the 3-D wave step by step on a ragged box
        dict(name="wave_ragged", kind="wave", variant="wave3d_f32", nx=201, ny=150, nz=97,
             kernel="proceed", per=1, steps=40, graph=False),
        # the misfit gradient of a wave rollout (two-step kernels and their adjoint)
        dict(name="wave_grad_192", kind="wave_grad", variant="wave3d_f32", nx=192, ny=192,
             nz=192, steps=20, every=10),
        # the wave in double precision
        dict(name="wave_f64_160", kind="wave", variant="wave3d_f64", nx=160, ny=160, nz=160,
             kernel="proceed", per=1, steps=20, graph=False),
    ]


def _log(rng, lo, hi):
    return int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))


def draw(rng):
    kind = rng.choice(["hydro", "hydro", "hydro64", "batch", "hydro_grad", "life", "life", "wave",
                       "wave", "wave64", "wave_grad"])
    graph = rng.random() < 0.5
    if kind in ("hydro", "hydro64"):
        hi = 2048 if kind == "hydro" else 1024
        return dict(kind="hydro", variant="hydro_f32" if kind == "hydro" else "hydro_f64",
                    nx=_log(rng, 48, hi), ny=_log(rng, 48, hi),
                    kernel=rng.choice(["proceed", "proceed_pipelined"]),
                    steps=rng.randint(8, 20), graph=graph)
    if kind == "batch":
        return dict(kind="batch", variant="hydro_f32_batch", grids=_log(rng, 8, 200), lo=64,
                    hi=_log(rng, 256, 1024), kernel="proceed_pipelined",
                    steps=rng.randint(10, 40), graph=graph)
    if kind == "hydro_grad":
        return dict(kind="hydro_grad", variant="hydro_adj2_f32_fast", nx=_log(rng, 64, 512),
                    ny=_log(rng, 64, 512), steps=rng.randint(10, 40), every=rng.randint(5, 20))
    if kind == "life":
        per = rng.choice([1, 4, 8])
        return dict(kind="life", variant="life_i32", nx=_log(rng, 64, 4096),
                    ny=_log(rng, 64, 4096), kernel="proceed" if per == 1 else "proceed_x%d" % per,
                    per=per, steps=rng.randint(20, 125), graph=graph)
    if kind == "wave_grad":
        return dict(kind="wave_grad", variant="wave3d_f32", nx=_log(rng, 32, 192),
                    ny=_log(rng, 32, 192), nz=_log(rng, 32, 192),
                    steps=2 * rng.randint(4, 12), every=2 * rng.randint(2, 6))
    per = 1 if kind == "wave64" else rng.choice([1, 2])
    hi = 384 if kind == "wave" else 192
    return dict(kind="wave", variant="wave3d_f32" if kind == "wave" else "wave3d_f64",
                nx=_log(rng, 32, hi), ny=_log(rng, 32, hi), nz=_log(rng, 32, hi),
                kernel="proceed" if per == 1 else "proceed_x2", per=per,
                steps=per * rng.randint(5, 20), graph=graph)


# ------------------------------------------------------------------ inputs
def _dtype(variant):
    return torch.float64 if variant.endswith("f64") else torch.float32


def _uniform(seed, *shape):
    g = torch.Generator(device="cuda").manual_seed(int(seed) & 0x7FFFFFFF)
    return torch.rand(shape, generator=g, device="cuda", dtype=torch.float64)


def _hydro_state(nx, ny, seed, dtype):
    """A Kelvin-Helmholtz flow some time after its start: two shear layers of finite width
    with a density contrast, a perturbation of seeded waves and a little noise."""
    x = ((torch.arange(nx, dtype=torch.float64, device="cuda") + 0.5) / nx)[None, :]
    y = ((torch.arange(ny, dtype=torch.float64, device="cuda") + 0.5) / ny)[:, None]
    r = _uniform(seed, 16).tolist()
    band = 0.5 * (torch.tanh((y - 0.25) / 0.04) - torch.tanh((y - 0.75) / 0.04))
    wave = sum((0.5 + r[k]) * torch.sin(2 * math.pi * ((k + 1) * x + r[k + 4]))
               * torch.cos(2 * math.pi * (y + r[k + 8])) for k in range(4))
    noise = _uniform(seed + 1, 4, ny, nx) - 0.5
    rho = 1.0 + band + 0.05 * wave + 0.02 * noise[0]
    v0 = band - 0.5 + 0.05 * wave + 0.02 * noise[1]
    v1 = 0.2 * wave + 0.02 * noise[2]
    p = 2.5 + 0.1 * wave + 0.02 * noise[3]
    return [f.to(dtype).contiguous() for f in (rho, v0, v1, p)]


def _wave_state(nx, ny, nz, seed, dtype):
    """Three seeded Gaussian pulses, eight cells wide (less in small boxes), and their rates."""
    out = []
    for part in range(2):
        f = torch.zeros((nz, ny, nx), dtype=torch.float64, device="cuda")
        u = _uniform(seed + part, 3, 4).tolist()
        for k in range(3):
            g = None
            for a, n in enumerate((nz, ny, nx)):
                d = torch.arange(n, dtype=torch.float64, device="cuda") - u[k][a] * n
                d = (d + n / 2.0) % n - n / 2.0
                e = torch.exp(-d * d / (2.0 * min(8.0, n / 8.0) ** 2))
                e = e.reshape([n if b == a else 1 for b in range(3)])
                g = e if g is None else g * e
            f += (0.5 + u[k][3]) * (1.0 if part == 0 else 0.1) * g
        out.append(f.to(dtype).contiguous())
    return out


def _life_state(nx, ny, seed):
    return (_uniform(seed, ny, nx) < 0.5).to(torch.int32).contiguous()


def _sizes(case, seed):
    """The uneven grids of a batch: the same for every seed, so that only values differ."""
    return [tuple(int(v) for v in s) for s in inputs.batched_sizes(case["grids"], 2024,
                                                                   case["lo"], case["hi"])]


DT = 1e-4                                       # of the differentiable, fixed-dt runs
COURANT = 0.5                                   # c dt / dx of the wave


def _square(nx, ny, dtype):
    x = (torch.arange(nx, dtype=torch.float64, device="cuda") + 0.5) / nx
    y = (torch.arange(ny, dtype=torch.float64, device="cuda") + 0.5) / ny
    return (((y >= 0.25) & (y <= 0.75))[:, None] & ((x >= 0.25) & (x <= 0.75))[None, :]).to(dtype)


# ------------------------------------------------------------------ the program's side
def _put(m, name, t):
    m.write_device(name, t.data_ptr(), t.numel() * t.element_size())


def _take(m, name, t):
    m.read_device(name, t.data_ptr(), t.numel() * t.element_size())


def prepare(case, seed):
    kind, dt = case["kind"], _dtype(case["variant"])
    if kind == "batch":
        sizes = _sizes(case, seed)
        b = variants.batch(case["variant"], sizes)
        cells = sum(nx * ny for nx, ny in sizes)
        outs = [torch.empty(cells, dtype=dt, device="cuda") for _ in HYDRO]
        for g, (nx, ny) in enumerate(sizes):
            for k, v in inputs.hydro_scalars(nx, ny).items():
                b.grids[g].set(k, v)
            fields = _hydro_state(nx, ny, seed + 2 * g, dt)
            torch.cuda.synchronize()
            for f, t in zip(HYDRO, fields):
                _put(b.grids[g], f, t)
            b.sync()
        b.run("proceed_prime")
        b.sync()
        return dict(case=case, batch=b, sizes=sizes, outs=outs)
    shape = [case[k] for k in ("nx", "ny", "nz") if k in case]
    m = variants.machine(case["variant"], shape)
    if kind in ("hydro", "hydro_grad"):
        for k, v in inputs.hydro_scalars(*shape).items():
            m.set(k, v)
        fields, names = _hydro_state(*shape, seed, dt), HYDRO
        if kind == "hydro_grad":
            m.set("dt", DT)
    elif kind == "life":
        m.run("init")
        fields, names = [_life_state(*shape, seed)], ("cell",)
    else:
        for k, v in (("c", 1.0), ("dx", 1.0), ("dt", COURANT)):
            m.set(k, v)
        fields, names = _wave_state(*shape, seed, dt), ("fieldF", "fieldG")
    torch.cuda.synchronize()
    m.sync()
    state = dict(case=case, m=m, names=names)
    if kind == "hydro_grad":
        state.update(fields=[f.requires_grad_() for f in fields], mask=_square(*shape, dt))
    elif kind == "wave_grad":
        state.update(fields=[f.requires_grad_() for f in fields],
                     target=_wave_state(*shape, seed + 7, dt)[0])
    else:
        for n, t in zip(names, fields):
            _put(m, n, t)
        if case["kernel"] == "proceed_pipelined":
            m.run("proceed_prime")
        m.sync()
        state["outs"] = fields
        if kind == "hydro":
            state["time"] = torch.zeros(1, dtype=dt, device="cuda")
        if kind == "life":
            state["population"] = torch.zeros(1, dtype=torch.int32, device="cuda")
    torch.cuda.synchronize()
    return state


def run(state):
    case = state["case"]
    kind = case["kind"]
    if kind == "hydro_grad":
        out = rollout(state["m"], HYDRO, state["fields"], case["steps"], case["every"],
                      fwd=["proceed_stage1", "proceed_stage2"],
                      adj=["proceed_stage2_adjoint", "proceed_stage1_adjoint"], tape_after=1)
        rho, v0, v1, _ = out
        objective = (0.5 * rho * (v0 * v0 + v1 * v1) * state["mask"]).sum()
        grads = torch.autograd.grad(objective, state["fields"])
        return {"fields": [o.detach() for o in out], "grads": list(grads)}
    if kind == "wave_grad":
        out = rollout(state["m"], state["names"], state["fields"], case["steps"] // 2,
                      case["every"] // 2, fwd="proceed_x2", adj="proceed_adjoint_x2")
        misfit = 0.5 * (out[0] - state["target"]).square().sum()
        grads = torch.autograd.grad(misfit, state["fields"])
        return {"fields": [o.detach() for o in out], "grads": list(grads)}
    if kind == "batch":
        b = state["batch"]
        b.run(case["kernel"], case["steps"], graph=case["graph"])
        at = 0
        for g, (nx, ny) in enumerate(state["sizes"]):
            for f, t in zip(HYDRO, state["outs"]):
                b.grids[g].read_device(f, t.data_ptr() + at * t.element_size(),
                                       nx * ny * t.element_size())
            at += nx * ny
        return {"fields": state["outs"]}
    m = state["m"]
    m.run(case["kernel"], case["steps"] // case.get("per", 1) if kind == "wave" else case["steps"],
          graph=case["graph"])
    for n, t in zip(state["names"], state["outs"]):
        _take(m, n, t)
    out = {"fields": state["outs"]}
    for n in ("time", "population"):
        if n in state:
            _take(m, n, state[n])
            out[n] = state[n]
    return out


def _cells(case):
    if case["kind"] == "batch":
        return sum(nx * ny for nx, ny in _sizes(case, 0))
    return case["nx"] * case["ny"] * case.get("nz", 1)


def work(case):
    """The state in and out once (with the gradients, where asked for), and the scheme's own
    operations on every cell and step (a reverse sweep: twice the forward's, and its replay)."""
    kind, cells = case["kind"], _cells(case)
    size = torch.empty(0, dtype=_dtype(case["variant"])).element_size()
    base = kind.split("_")[0].replace("batch", "hydro")
    fields = {"hydro": 4, "life": 1, "wave": 2}[base]
    steps = case["steps"] * (case["per"] if kind == "life" else 1)
    ops = OPS[base] * cells * steps
    if kind == "hydro_grad":
        return {"bytes": 3 * fields * size * cells, "flops": 4 * ops}
    if kind == "wave_grad":       # linear: no replay
        return {"bytes": (3 * fields + 1) * size * cells, "flops": 2 * ops}
    return {"bytes": 2 * fields * size * cells, "flops": ops}


# ------------------------------------------------------------------ the same in 64 bits
def _rounded(x, variant):
    return float(np.float32(x)) if _dtype(variant) is torch.float32 else float(x)


class _Gas:
    """A state with its derived quantities, from rho, v, p or from rho, momentum, energy."""

    def __init__(self, rho, v=None, p=None, m=None, e=None):
        self.rho = rho
        if v is not None:
            self.v, self.p = list(v), p
            self.m = [rho * a for a in self.v]
            self.e = 0.5 * (self.v[0] * self.m[0] + self.v[1] * self.m[1]) + p / (GAMMA - 1)
        else:
            self.m, self.e = list(m), e
            self.v = [a / rho for a in self.m]
            self.p = (GAMMA - 1) * (e - 0.5 * (self.v[0] * self.m[0] + self.v[1] * self.m[1]))

    def sound(self):
        return torch.sqrt(GAMMA * self.p / self.rho)

    def flux(self, i):
        m = [self.m[j] * self.v[i] + (self.p if j == i else 0.0) for j in range(2)]
        return [self.m[i]] + m + [(self.e + self.p) * self.v[i]]


def _at(a, n, axis):
    return torch.roll(a, n, 1 - axis)


def _faces(order, i, s):
    def sides(a):
        a1 = _at(a, 1, i)
        if order == 1:
            return a1, a
        d0, d1, d2 = a1 - _at(a, 2, i), a - a1, _at(a, -1, i) - a

        def limited(u, w):
            return torch.where(u * w <= 0, torch.zeros_like(u), torch.where(u.abs() < w.abs(), u, w))
        return a1 + limited(d0, d1) / 2, a - limited(d1, d2) / 2
    (rl, rr), (ul, ur), (wl, wr), (pl, pr) = (sides(a) for a in (s.rho, s.v[0], s.v[1], s.p))
    return _Gas(rl, (ul, wl), pl), _Gas(rr, (ur, wr), pr)


def _riemann(i, L, R):
    cl, cr = L.sound(), R.sound()
    ul, ur = L.v[i], R.v[i]
    star = torch.clamp((L.p + R.p) / 2 - (L.rho + R.rho) / 2 * ((cl + cr) / 2) * (ur - ul), min=0)

    def q(p):
        return torch.where(p <= star, torch.ones_like(p),
                           torch.sqrt(1 + (GAMMA + 1) / (2 * GAMMA) * (star / p - 1)))
    sl, sr = ul - cl * q(L.p), ur + cr * q(R.p)
    al, ar = L.rho * (sl - ul), R.rho * (sr - ur)
    mid = (R.p - L.p + al * ul - ar * ur) / (al - ar)

    def between(s, w):
        u = w.v[i]
        rho = w.rho * (s - u) / (s - mid)
        m = [rho * (mid if j == i else w.v[j]) for j in range(2)]
        return _Gas(rho, m=m, e=rho * (w.e / w.rho + (mid - u) * (mid + w.p / w.rho / (s - u))))
    parts = [w.flux(i) for w in (L, between(sl, L), between(sr, R), R)]
    return [torch.where(sl > 0, a, torch.where(mid > 0, b, torch.where(sr > 0, c, d)))
            for a, b, c, d in zip(*parts)]


def _half(order, dt, d, s, base):
    rho, m, e = base.rho, list(base.m), base.e
    fx = [_riemann(i, *_faces(order, i, s)) for i in range(2)]
    g = base
    for i in (1, 0):
        df = [f - _at(f, -1, i) for f in fx[i]]
        g = _Gas(g.rho + dt / d[i] * df[0], m=[g.m[j] + dt / d[i] * df[1 + j] for j in range(2)],
                 e=g.e + dt / d[i] * df[3])
    return _Gas(torch.clamp(g.rho, min=1e-2), g.v, torch.clamp(g.p, min=1e-2))


def _hydro_steps(fields, steps, d, cfl=None, dt=None):
    time = 0.0
    for _ in range(steps):
        s = _Gas(fields[0], fields[1:3], fields[3])
        if cfl is not None:
            c = s.sound()
            dt = cfl * torch.minimum(d[0] / (c + s.v[0].abs()), d[1] / (c + s.v[1].abs())).min()
        s = _half(2, dt, d, _half(1, dt / 2, d, s, s), s)
        fields, time = [s.rho, s.v[0], s.v[1], s.p], time + dt
    return fields, time


def _wave_steps(f, g, steps):
    for _ in range(steps):
        f = f + COURANT * g
        lap = sum(torch.roll(f, 1, a) + torch.roll(f, -1, a) - 2 * f for a in range(3))
        g = g + COURANT * lap
    return f, g


def exact(case, seed):
    kind, dtype = case["kind"], _dtype(case["variant"])
    if kind in ("hydro", "hydro_grad"):
        nx, ny = case["nx"], case["ny"]
        fields = [f.double() for f in _hydro_state(nx, ny, seed, dtype)]
        d = [_rounded(1.0 / nx, case["variant"]), _rounded(1.0 / ny, case["variant"])]
        if kind == "hydro":
            out, time = _hydro_steps(fields, case["steps"], d, cfl=_rounded(0.4, case["variant"]))
            return {"fields": out, "time": time.reshape(1)}
        fields = [f.requires_grad_() for f in fields]
        out, _ = _hydro_steps(fields, case["steps"], d, dt=_rounded(DT, "f32"))
        objective = (0.5 * out[0] * (out[1] ** 2 + out[2] ** 2) * _square(nx, ny, torch.float64)).sum()
        return {"fields": [o.detach() for o in out],
                "grads": list(torch.autograd.grad(objective, fields))}
    if kind == "batch":
        outs = [[] for _ in HYDRO]
        for g, (nx, ny) in enumerate(_sizes(case, seed)):
            d = [_rounded(1.0 / nx, case["variant"]), _rounded(1.0 / ny, case["variant"])]
            fields = [f.double() for f in _hydro_state(nx, ny, seed + 2 * g, dtype)]
            out, _ = _hydro_steps(fields, case["steps"], d, cfl=_rounded(0.4, case["variant"]))
            for o, f in zip(outs, out):
                o.append(f.reshape(-1))
        return {"fields": [torch.cat(o) for o in outs]}
    if kind == "life":
        cell = _life_state(case["nx"], case["ny"], seed)
        for _ in range(case["steps"] * case["per"]):
            n = sum(torch.roll(cell, (a, b), (0, 1)) for a in (-1, 0, 1) for b in (-1, 0, 1)) - cell
            cell = ((n == 3) | ((cell == 1) & (n == 2))).to(torch.int32)
        return {"fields": [cell], "population": cell.sum().to(torch.int32).reshape(1)}
    f, g = (t.double() for t in _wave_state(case["nx"], case["ny"], case["nz"], seed, dtype))
    if kind == "wave":
        return {"fields": list(_wave_steps(f, g, case["steps"]))}
    target = _wave_state(case["nx"], case["ny"], case["nz"], seed + 7, dtype)[0].double()
    f, g = f.requires_grad_(), g.requires_grad_()
    out = _wave_steps(f, g, case["steps"])
    misfit = 0.5 * (out[0] - target).square().sum()
    return {"fields": [o.detach() for o in out], "grads": list(torch.autograd.grad(misfit, (f, g)))}
