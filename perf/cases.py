"""The work a user of this framework has it do, as cases that can be timed.

A case is one call path through the public entry points (``hype2d.Context``,
``Batch``, ``Server``, ``rhs_noalloc`` and the C ABI's device-buffer forms),
with its system, path, order, boundaries and grid.  ``listed`` names the cases,
``draw`` gives more of the same ranges, ``prepare`` makes what a program holds
before the call, ``run`` makes one pass, ``work`` says what that pass cannot do
without, and ``exact`` computes the same outputs in plain torch, in 64 bits.

The kinds of call:

* ``rhs``    the right-hand side on device buffers, as a time integrator that
             keeps its vectors on the GPU calls it at every stage;
* ``noalloc`` the same on caller-owned buffers without a context;
* ``host``   the right-hand side on host buffers: the drop-in for a PETSc
             program whose vectors live in host memory;
* ``prim``   the primitive pass that snapshots and restarts are written from;
* ``solve``  a device-resident SSP-RK solve: set the state, step, read it back;
* ``batch``  many grids of one study advanced together;
* ``served`` a queue of solve requests of mixed systems and sizes, drained.

Grids range from 48 cells a side (coarse studies, the served mix's smallest)
to the 2048 x 1024 of the water-air problem; states are the shock-bubble,
four-quadrant, water-air and smooth periodic fields those systems are run on,
with strengths, radii and positions drawn from the seed.
"""
import ctypes
import math
import os
import random
import sys

import numpy as np
import torch

sys.path.insert(0, os.path.join(os.path.dirname(os.path.dirname(os.path.abspath(__file__))), "hype-parallel_amd"))
import hype2d as H  # noqa: E402

SYSTEMS = {"euler": H.EULER, "kapila": H.KAPILA, "bn": H.BAER_NUNZIATO}
NVAR = {"euler": 4, "kapila": 6, "bn": 9}
BC = {"I": H.BC_INLET, "P": H.BC_PERIODIC, "R": H.BC_REFLECTIVE, "T": H.BC_TRANSMISSIVE}
STAGES = {1: 2, 2: 4, 3: 10}  # SSPRK(2,2), SSPRK(4,3), SSPRK(10,4)
CFL = 0.5


def case(name, kind, system, nx, ny, *, prim=True, order=2, bc="TTTT", fma=False, steps=0, count=1, lo=0):
    c = {"name": name} if name else {}
    return {**c, "kind": kind, "system": system, "nx": nx, "ny": ny, "prim": prim, "order": order, "bc": bc,
            "fma": fma, "steps": steps, "count": count, "lo": lo}


def listed():
    return [
        # a coarse grid: launch latency and the host side of one callback
        case("rhs_euler_64x64", "rhs", "euler", 64, 64),
        # a ragged mid-size grid with walls, called once per stage by an outer integrator
        case("rhs_kapila_517x301", "rhs", "kapila", 517, 301, bc="TTRR"),
        # the context-free callback, on the other path of the largest system
        case("noalloc_bn_prim_333x260", "noalloc", "bn", 333, 260, bc="TTRT"),
        # the drop-in for a host-memory PETSc program: both transfers are part of the call
        case("host_kapila_1024x512", "host", "kapila", 1024, 512, bc="TTRR"),
        # primitive variables of the largest grid, for a snapshot
        case("prim_bn_2048x1024", "prim", "bn", 2048, 1024, prim=False),
        # the four-quadrant problem: a small grid stepped many times
        case("solve_euler_256x256", "solve", "euler", 256, 256, steps=20),
        # minmod slopes on the conservative path, a fine odd grid
        case("solve_euler_cons_minmod_1535x1023", "solve", "euler", 1535, 1023, prim=False, order=1, bc="RRRR", steps=4),
        # the shock-bubble
        case("solve_kapila_1024x512", "solve", "kapila", 1024, 512, bc="TTRR", steps=10),
        # the periodic vortex study's highest order, at a middle refinement
        case("solve_kapila_order3_256x256", "solve", "kapila", 256, 256, order=3, bc="PPPP", steps=3),
        # the water-air interface, the largest single grid
        case("solve_bn_cons_2048x1024", "solve", "bn", 2048, 1024, prim=False, steps=3),
        # a parameter study: shock-bubbles of sides 128 to 1024 advanced together
        case("batch_kapila_48_of_128_to_1024", "batch", "kapila", 1024, 1024, bc="TTRR", steps=2, count=48, lo=128),
        # a served queue of all three systems, half of it with the contracted kernels allowed
        case("served_mix_16_of_64_to_512", "served", "mix", 512, 512, steps=12, count=16, lo=64, fma=True),
    ]


def _side(rng, lo, hi):
    return int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))


def draw(rng):
    kind = rng.choice(["rhs", "rhs", "noalloc", "host", "prim", "solve", "solve", "solve", "batch", "served"])
    if kind == "served":
        return case(None, "served", "mix", 512, 512, steps=rng.randint(6, 12), count=rng.randint(6, 16),
                    lo=_side(rng, 48, 128), fma=rng.random() < 0.5)
    system = rng.choice(["euler", "kapila", "kapila", "bn"])
    order = rng.choice([1, 2, 2, 2, 3])
    prim = rng.random() < 0.65
    if kind == "batch":
        return case(None, "batch", system, 512, 512, prim=prim, order=order, bc="TTRR", steps=2,
                    count=rng.randint(8, 40), lo=_side(rng, 64, 200), fma=rng.random() < 0.2)
    nx, ny = _side(rng, 48, 2048), _side(rng, 48, 1024)
    bc = rng.choice(["TTTT", "TTRR", "RRTT", "PPPP", "PPRT"])
    if system == "kapila" and order < 3 and rng.random() < 0.2:
        bc = "ITRR"
    if order == 3:
        bc = "PPPP"
    steps = 0
    if kind == "solve":
        steps = max(1, min(20, int(2.0e7 / (nx * ny * NVAR[system] * STAGES[order]))))
    return case(None, kind, system, nx, ny, prim=prim, order=order, bc=bc,
                fma=kind in ("rhs", "solve") and rng.random() < 0.2, steps=steps)


# --------------------------------------------------------------- states ----
EOS = {"euler": (1.4, 1.4, 0.0, 0.0), "kapila": (1.4, 1.648, 0.0, 0.0), "bn": (4.4, 1.4, 6.0e8, 0.0)}
JET = (4.4, 1.4, 6000.0, 0.0)  # water-air constants of the inlet runs


def _grids(c, seed):
    """The grids of a case: dicts with system, nx, ny, prim, order, bc, fma, eos, seed, domain."""
    rng = random.Random(seed)
    out = []
    for k in range(c["count"]):
        g = {n: c[n] for n in ("system", "nx", "ny", "prim", "order", "bc", "fma")}
        if c["kind"] in ("batch", "served"):  # sizes are the case's, not the seed's
            sizes = random.Random(1000 * c["count"] + c["lo"] + k)
            g["nx"] = _side(sizes, c["lo"], c["nx"])
            g["ny"] = g["nx"] if c["kind"] == "served" else _side(sizes, c["lo"], c["ny"])
            if c["system"] == "mix":
                g["system"] = ("euler", "kapila", "euler", "kapila", "bn")[k % 5]
                g["prim"] = g["system"] != "bn"
                g["bc"] = "TTRR" if g["system"] == "kapila" else "TTTT"
                g["fma"] = c["fma"] and k % 2 == 1
        g["eos"] = JET if g["bc"][0] == "I" else EOS[g["system"]]
        g["seed"] = rng.randrange(1 << 30)
        h = (30.0 if g["bc"][0] == "I" else 1.0) / g["ny"]
        y0 = -15.0 if g["bc"][0] == "I" else 0.0
        g["domain"] = (0.0, g["nx"] * h, y0, y0 + g["ny"] * h)
        out.append(g)
    return out


def _problem(g):
    g1, g2, p1, p2 = g["eos"]
    return H.make_problem(SYSTEMS[g["system"]], g["nx"], g["ny"], order=g["order"], prim=g["prim"],
                          domain=g["domain"], cfl=CFL, bc=tuple(BC[b] for b in g["bc"]), gamma1=g1, gamma2=g2,
                          pi1=p1, pi2=p2, fma=g["fma"])


def _state(g, device):
    """Conserved cell values, shape (ny, nx, nvar), of the grid's problem."""
    rng = random.Random(g["seed"])
    x0, x1, y0, y1 = g["domain"]
    f64 = {"dtype": torch.float64, "device": device}
    h = (x1 - x0) / g["nx"]
    x = (x0 + h * (torch.arange(g["nx"], **f64) + 0.5))[None, :].expand(g["ny"], g["nx"])
    y = (y0 + h * (torch.arange(g["ny"], **f64) + 0.5))[:, None].expand(g["ny"], g["nx"])
    lx = x1 - x0
    one = torch.ones_like(x)
    g1, g2, p1, p2 = g["eos"]
    smooth = g["bc"] == "PPPP"
    if g["system"] == "euler":
        if smooth:  # an entropy and pressure wave pair carried diagonally
            a, ph = rng.uniform(0.1, 0.3), rng.uniform(0, 6)
            kx, ky = 2 * math.pi / lx, 2 * math.pi
            rho = 1 + a * torch.sin(kx * x + 2 * ky * y + ph)
            u, v, p = 0.7 + 0.1 * torch.sin(ky * y), -0.4 * one, 1 + 0.1 * torch.cos(kx * x - ph)
        else:  # four quadrants
            right, top = x >= lx * rng.uniform(0.35, 0.65), y >= rng.uniform(0.35, 0.65)
            q = [[v * rng.uniform(0.95, 1.05) for v in s] for s in ((1.5, 0.0, 0.0, 1.5), (0.5323, 1.206, 0.0, 0.3),
                                                                    (0.138, 1.206, 1.206, 0.029), (0.5323, 0.0, 1.206, 0.3))]
            rho, u, v, p = (torch.where(right, torch.where(top, q[0][k] * one, q[3][k] * one),
                                        torch.where(top, q[1][k] * one, q[2][k] * one)) for k in range(4))
        return torch.stack([rho, rho * u, rho * v, p / (g1 - 1) + 0.5 * rho * (u * u + v * v)], -1).contiguous()
    if g["system"] == "kapila":
        if g["bc"][0] == "I":  # a jet entering still water
            r1, r2, u, v = 1000.0 * one, one, 0 * one, 0 * one
            p = 1.013 * (1 + 0.01 * torch.sin(0.3 * y + rng.uniform(0, 6)))
            a = (1 - 1e-6) * one
        elif smooth:  # a diffuse interface in a uniform stream
            ph = rng.uniform(0, 6)
            r = torch.hypot(x - 0.5 * lx, y - 0.5)
            r1 = 1.4 + 0.1 * torch.sin(2 * math.pi * (x / lx + y) + ph)
            r2 = 0.25463 * (1 + 0.1 * torch.cos(2 * math.pi * (x / lx - y)))
            u, v, p = 100 * one, 60 * one, 1e5 * one
            a = 0.25 + 0.25 * torch.erfc((r / rng.uniform(0.2, 0.3) - 1) / 0.3)
        else:  # a shock running into a helium bubble
            mach, rad = rng.uniform(1.1, 2.0), rng.uniform(0.1, 0.3)
            cx, cy, xs = lx * rng.uniform(0.4, 0.6), rng.uniform(0.4, 0.6), lx * rng.uniform(0.05, 0.1)
            r = torch.hypot(x - cx, y - cy)
            a = 1e-6 + (1 - 2e-6) * 0.5 * (1 + torch.tanh((r - rad) / (2 * h)))
            hit = x < xs
            p_post = 1e5 * (1 + 2 * g1 / (g1 + 1) * (mach * mach - 1))
            r_post = 1.4 * (g1 + 1) * mach * mach / ((g1 - 1) * mach * mach + 2)
            u_post = mach * math.sqrt(g1 * 1e5 / 1.4) * (1 - 1.4 / r_post)
            r1 = torch.where(hit, r_post * one, 1.4 * one)
            r2, v = 0.25463 * one, 0 * one
            u, p = torch.where(hit, u_post * one, 0 * one), torch.where(hit, p_post * one, 1e5 * one)
        rho = a * r1 + (1 - a) * r2
        en = a * (p + g1 * p1) / (g1 - 1) + (1 - a) * (p + g2 * p2) / (g2 - 1)
        return torch.stack([a * r1, (1 - a) * r2, rho * u, rho * v, en + 0.5 * rho * (u * u + v * v), a], -1).contiguous()
    # Baer-Nunziato: water below a wavy interface, air above, a burst of pressure
    eta = 0.5 + 0.03 * torch.sin(2 * math.pi * rng.randint(1, 4) * x / lx + rng.uniform(0, 6))
    a = 1e-6 + (1 - 2e-6) * 0.5 * (1 - torch.tanh((y - eta) / (2 * h)))
    burst = torch.hypot(x - lx * rng.uniform(0.4, 0.6), y - rng.uniform(0.2, 0.3)) < rng.uniform(0.08, 0.12)
    p = torch.where(burst, rng.uniform(2e8, 1e9) * one, 1e5 * one)
    r1, r2 = 1000.0 * one, one
    m1, m2 = a * r1, (1 - a) * r2
    e1, e2 = (p + g1 * p1) / (r1 * (g1 - 1)), (p + g2 * p2) / (r2 * (g2 - 1))
    zero = torch.zeros_like(x)
    return torch.stack([m1, zero, zero, m1 * e1, m2, zero, zero, m2 * e2, a], -1).contiguous()


# ------------------------------------------------------------ the passes ----
def _ptr(t):
    return ctypes.cast(t.data_ptr(), ctypes.POINTER(ctypes.c_double))


def prepare(case, seed):
    kind = case["kind"]
    grids = _grids(case, seed)
    s = {"kind": kind, "grids": grids, "steps": case["steps"]}
    states = [_state(g, "cuda") for g in grids]
    problems = [_problem(g) for g in grids]
    if kind == "served":
        s["requests"] = [(p, U.cpu().numpy()) for p, U in zip(problems, states)]
        s["server"] = H.Server()
        return s
    if kind == "batch":
        s["batch"] = H.Batch(problems)
    elif kind != "noalloc":
        s["ctx"] = H.Context(problems[0])
    s["problem"] = problems[0]
    if kind == "host":
        s["U"] = states[0].cpu().numpy()
        return s
    s["U"] = states
    s["out"] = [torch.empty_like(U) for U in states]
    torch.cuda.synchronize()  # the framework works on streams of its own
    return s


def run(state):
    kind = state["kind"]
    if kind == "host":
        rhs, dt, _ = state["ctx"].rhs(state["U"])
        return {"rhs": rhs, "dt": dt}
    if kind == "served":
        srv = state["server"]
        ids = [srv.submit(p, U, max_steps=state["steps"]) for p, U in state["requests"]]
        srv.drain()
        done = [srv.result(i) for i in ids]
        return {"U": [U for U, _ in done], "steps": np.array([info.status.steps for _, info in done]),
                "t": np.array([info.status.t for _, info in done])}
    U, out = state["U"], state["out"]
    if kind == "rhs":
        dt = state["ctx"].rhs_device(U[0].data_ptr(), out[0].data_ptr())
        return {"rhs": out[0], "dt": dt}
    if kind == "noalloc":
        dt, _, _ = H.rhs_noalloc(state["problem"], U[0].data_ptr(), out[0].data_ptr())
        return {"rhs": out[0], "dt": dt}
    lib = H.lib()

    def ok(rc):
        if rc != H.OK:
            raise H.HypeError(rc, kind)

    if kind == "prim":
        ok(lib.hype_cons2prim(state["ctx"].h, _ptr(U[0]), _ptr(out[0]), H.MEM_DEVICE))
        return {"W": out[0]}
    if kind == "solve":
        ctx = state["ctx"]
        ok(lib.hype_set_state(ctx.h, _ptr(U[0]), H.MEM_DEVICE))
        ctx.begin(max_steps=state["steps"], flags=H.TS_CLIP | H.TS_GRAPH)
        ctx.advance(state["steps"])
        st = ctx.sync()
        ok(lib.hype_get_state(ctx.h, _ptr(out[0]), H.MEM_DEVICE))
        return {"U": out[0], "steps": st.steps, "t": st.t}
    b = state["batch"]
    for i in range(len(b)):
        ok(lib.hype_batch_set_state(b.h, i, _ptr(U[i]), H.MEM_DEVICE))
    b.begin(max_steps=state["steps"])
    b.advance(state["steps"])
    sts = b.sync()
    for i in range(len(b)):
        ok(lib.hype_batch_get_state(b.h, i, _ptr(out[i]), H.MEM_DEVICE))
    return {"U": list(out), "steps": np.array([st.steps for st in sts]), "t": np.array([st.t for st in sts])}


def work(case):
    """Each state once in and once out per stage (one more read of the step's
    start where the scheme combines with it), and the arithmetic of one
    right-hand side per cell, an operation each for +, -, *, / and sqrt."""
    byts = flops = 0.0
    for g in _grids(case, 0):
        n, nv = g["nx"] * g["ny"], NVAR[g["system"]]
        order = g["order"]
        recon = {1: 12, 2: 194, 3: 330}[order] * nv          # slopes or weights and coefficients
        points = {1: 4, 2: 8, 3: 8}[order]
        values = points * {1: 4, 2: 10, 3: 18}[order] * nv   # values at the face points
        face = {"euler": 60, "kapila": 150, "bn": 170}[g["system"]] * points // 2
        volume = {"euler": 0, "kapila": 90, "bn": 60}[g["system"]] * (1 if order == 1 else 4)
        per = recon + values + face + volume + 10 * nv
        if case["kind"] == "prim":
            byts += 16.0 * nv * n
            flops += {"euler": 13, "kapila": 24, "bn": 30}[g["system"]] * n
            continue
        stages = case["steps"] * STAGES[order] if case["steps"] else 1
        passes = case["steps"] * {1: 5, 2: 9, 3: 22}[order] if case["steps"] else 2
        byts += 8.0 * nv * n * passes
        flops += float(per) * n * (stages + (1 if case["steps"] else 0))
    return {"bytes": byts, "flops": flops}


# ------------------------------------------- the same in plain torch, 64 bits
def exact(case, seed):
    device = "cuda" if torch.cuda.is_available() else "cpu"
    kind = case["kind"]
    done = []
    for g in _grids(case, seed):
        U = _state(g, device)
        if kind == "prim":
            return {"W": torch.stack(_to_prim(g, list(U.unbind(-1))), -1)}
        if kind in ("rhs", "noalloc", "host"):
            rhs, dt = _rhs(g, U)
            return {"rhs": rhs.cpu().numpy() if kind == "host" else rhs, "dt": dt}
        done.append(_solve(g, U, case["steps"]))
    t = [d[1] for d in done]
    if kind == "solve":
        return {"U": done[0][0], "steps": None, "t": t[0]}
    states = [d[0].cpu().numpy() if kind == "served" else d[0] for d in done]
    return {"U": states, "steps": None, "t": np.array(t)}


def _solve(g, U, steps):
    """The SSP Runge-Kutta scheme of the order; dt of a step comes from the
    wave speeds of the last right-hand side of the step before."""
    t = 0.0
    _, dt = _rhs(g, U)
    for _ in range(steps):
        w = U
        if g["order"] == 1:
            w = w + dt * _rhs(g, w)[0]
            L, dt_next = _rhs(g, w)
            U = 0.5 * w + dt / 2 * L + 0.5 * U
        elif g["order"] == 2:
            for _ in range(2):
                w = w + dt / 2 * _rhs(g, w)[0]
            w = (2.0 / 3.0) * U + dt / 6 * _rhs(g, w)[0] + (1.0 / 3.0) * w
            L, dt_next = _rhs(g, w)
            U = w + dt / 2 * L
        else:
            for _ in range(5):
                w = w + dt / 6 * _rhs(g, w)[0]
            w1 = 0.04 * U + 0.36 * w
            w = 15.0 * w1 - 5.0 * w
            for _ in range(4):
                w = w + dt / 6 * _rhs(g, w)[0]
            L, dt_next = _rhs(g, w)
            U = 0.6 * w + dt / 10 * L + w1
        t, dt = t + dt, dt_next
    return U, t


def _to_prim(g, q):
    g1, g2, p1, p2 = g["eos"]
    if g["system"] == "euler":
        ir = 1.0 / q[0]
        return [q[0], ir * q[1], ir * q[2], (g1 - 1.0) * (q[3] - 0.5 * ir * (q[1] * q[1] + q[2] * q[2]))]
    if g["system"] == "kapila":
        a, b = q[5], 1.0 - q[5]
        rho = q[0] + q[1]
        u, v = q[2] / rho, q[3] / rho
        en = q[4] - 0.5 * rho * (u * u + v * v)
        p = (en * (g1 - 1.0) * (g2 - 1.0) - a * g1 * p1 * (g2 - 1.0) - b * g2 * p2 * (g1 - 1.0)) / (a * (g2 - 1.0) + b * (g1 - 1.0))
        return [q[0] / a, q[1] / b, u, v, p, a]
    out = []
    for a, k, gm, pi in ((q[8], 0, g1, p1), (1.0 - q[8], 4, g2, p2)):
        r, u, v = q[k] / a, q[k + 1] / q[k], q[k + 2] / q[k]
        out += [r, u, v, (gm - 1.0) * (q[k + 3] / a - 0.5 * r * (u * u + v * v)) - gm * pi]
    return out + [q[8]]


def _to_cons(g, w):
    g1, g2, p1, p2 = g["eos"]
    if g["system"] == "euler":
        r, u, v, p = w
        return [r, r * u, r * v, 0.5 * r * (u * u + v * v) + p / (g1 - 1.0)]
    if g["system"] == "kapila":
        r1, r2, u, v, p, a = w
        b = 1.0 - a
        rho = a * r1 + b * r2
        en = (p * (a * (g2 - 1.0) + b * (g1 - 1.0)) + a * g1 * p1 * (g2 - 1.0) + b * g2 * p2 * (g1 - 1.0)) / ((g1 - 1.0) * (g2 - 1.0))
        return [a * r1, b * r2, rho * u, rho * v, en + 0.5 * rho * (u * u + v * v), a]
    out = []
    for a, k, gm, pi in ((w[8], 0, g1, p1), (1.0 - w[8], 4, g2, p2)):
        r, u, v, p = w[k:k + 4]
        m = a * r
        out += [m, m * u, m * v, m * (0.5 * (u * u + v * v) + (p + gm * pi) / (r * (gm - 1.0)))]
    return out + [w[8]]


def _sound(g, w):
    """Kapila: rho_k a_k^2 of the phases and the mixture's squared speed of sound."""
    g1, g2, p1, p2 = g["eos"]
    r1, r2, a, b = w[0], w[1], w[5], 1.0 - w[5]
    a1, a2 = g1 * (w[4] + p1) / r1, g2 * (w[4] + p2) / r2
    rho = a * r1 + b * r2
    return r1 * a1, r2 * a2, (r1 * a1 * r2 * a2) / (rho * (b * r1 * a1 + a * r2 * a2))


def _admissible(g, w):
    """The check at a reconstructed point, on the path's own variables."""
    g1, g2, p1, p2 = g["eos"]
    if not g["prim"]:
        v = _to_prim(g, w)
        if g["system"] == "euler":
            return (v[0] >= 1e-14) & (v[3] >= 1e-12)
        if g["system"] == "kapila":  # this path's check asks for a pure phase 1
            return (w[5] == 1.0) & (_sound(g, v)[2] >= 1e-12)
        w = v
    if g["system"] == "euler":
        return (w[0] >= 1e-14) & (w[3] >= 1e-12)
    if g["system"] == "kapila":
        rho = w[5] * w[0] + (1.0 - w[5]) * w[1]
        return (rho >= 1e-14) & (_sound(g, w)[2] >= 1e-12) & (w[5] >= 0.0) & (w[5] <= 1.0)
    return ((w[0] >= 1e-14) & (w[4] >= 1e-14) & (w[3] + p1 >= 1e-12) & (w[7] + p2 >= 1e-12) & (w[8] >= 0.0) & (w[8] <= 1.0))


def _flux(g, x, axis):
    """(flux, wave speed, conserved state) across an axis from path variables x."""
    g1, g2, p1, p2 = g["eos"]
    w = x if g["prim"] else _to_prim(g, x)
    q = _to_cons(g, x) if g["prim"] else x
    if g["system"] == "euler":
        un, p = w[1 + axis], w[3]
        E = p / (g1 - 1.0) + 0.5 * w[0] * (w[1] * w[1] + w[2] * w[2]) if g["prim"] else q[3]
        f = [w[0] * un, w[0] * un * w[1], w[0] * un * w[2], un * (E + p)]
        f[1 + axis] = f[1 + axis] + p
        return f, un.abs() + torch.sqrt(g1 * p / w[0]), q
    if g["system"] == "kapila":
        un, p, a = w[2 + axis], w[4], w[5]
        b = 1.0 - a
        rho = a * w[0] + b * w[1] if g["prim"] else q[0] + q[1]
        f = [a * w[0] * un, b * w[1] * un, rho * w[2] * un, rho * w[3] * un, (q[4] + p) * un, torch.zeros_like(un)]
        f[2 + axis] = f[2 + axis] + p
        return f, un.abs() + torch.sqrt(_sound(g, w)[2]), q
    f, s = [], None
    for a, k, gm, pi in ((w[8], 0, g1, p1), (1.0 - w[8], 4, g2, p2)):
        r, u, v, p = w[k:k + 4]
        un = w[k + 1 + axis]
        E = (p + gm * pi) / (gm - 1.0) + 0.5 * r * (u * u + v * v) if g["prim"] else q[k + 3] / a
        part = [a * r * un, r * u * un, r * v * un, a * un * (E + p)]
        part[1 + axis] = part[1 + axis] + p
        f += [part[0], a * part[1], a * part[2], part[3]]
        speed = un.abs() + torch.sqrt(gm * (p + pi) / r)
        s = speed if s is None else torch.maximum(s, speed)
    return f + [torch.zeros_like(s)], s, q


def _nonconservative(g, x, dx, dy):
    """B(x) . grad by component (None where zero); dx, dy: gradients of the path variables."""
    if g["system"] == "euler":
        return [None] * 4
    w = x if g["prim"] else _to_prim(g, x)
    if g["system"] == "kapila":
        a, b = w[5], 1.0 - w[5]
        s1, s2, _ = _sound(g, w)
        K = a * b * (s2 - s1) / (a * s2 + b * s1)
        if g["prim"]:
            ux, vy = dx[2], dy[3]
        else:
            ir = 1.0 / (x[0] + x[1])
            rho = x[0] + x[1]
            ux = ir * ir * (dx[2] * rho - x[2] * (dx[0] + dx[1]))
            vy = ir * ir * (dy[3] * rho - x[3] * (dy[0] + dy[1]))
        return [None] * 5 + [w[2] * dx[5] + w[3] * dy[5] - K * (ux + vy)]
    p, n = w[7], w[1] * dx[8] + w[2] * dy[8]
    return [None, -p * dx[8], -p * dy[8], -p * n, None, p * dx[8], p * dy[8], p * n, n]


def _ghosted(g, planes):
    """Planes with a frame of three ghost cells on every side."""
    nx, ny, bc = g["nx"], g["ny"], g["bc"]
    flips = {"euler": ((1,), (2,)), "kapila": ((2,), (3,)), "bn": ((1, 5), (2, 6))}[g["system"]]

    def source(n, lo, hi):
        idx, sign = [], []
        for i in range(-3, n + 3):
            kind = lo if i < 0 else hi if i >= n else "-"
            j = {"-": i, "P": i % n, "I": i % n, "T": min(max(i, 0), n - 1), "R": -1 - i if i < 0 else 2 * n - 1 - i}[kind]
            idx.append(j)
            sign.append(-1.0 if kind == "R" else 1.0)
        return torch.tensor(idx, device=planes[0].device), torch.tensor(sign, dtype=torch.float64, device=planes[0].device)

    ix, sx = source(nx, bc[0], bc[1])
    iy, sy = source(ny, bc[2], bc[3])
    inlet = _inlet(g) if bc[0] == "I" else None
    out = []
    for c, a in enumerate(planes):
        a = a[:, ix]
        if inlet is not None:
            a[:, :3] = inlet[c].to(a.device)[3:-3, None]
        elif c in flips[0]:
            a = a * sx
        a = a[iy, :]
        out.append(a * sy[:, None] if c in flips[1] else a)
    return out


def _inlet(g):
    """The left inlet's state in path variables, by ghosted row (rows -3 .. ny + 2)."""
    h = (g["domain"][1] - g["domain"][0]) / g["nx"]
    speed = 2.0 * math.sqrt(g["eos"][1] * 1.013 / 1.0)
    mid, half, width = 0.5 * ((1.0 - 1.0e-6) + 1.0e-6), (1.0e-6 - (1.0 - 1.0e-6)) / 2.0, 3.0 * (30.0 / 500.0)
    rows = []
    for j in range(-3, g["ny"] + 3):
        y = g["domain"][2] + (j + 0.5) * h
        u = 2.0 * speed * (1.0 - y * y) if abs(y) < 1.0 else 0.0
        rows.append([1000.0, 1.0, u, 0.0, 1.013, mid + half * math.tanh(-(abs(y) - 1.0) / width)])
    w = list(torch.tensor(rows, dtype=torch.float64).unbind(-1))
    return w if g["prim"] else _to_cons(g, w)


def _minmod(a, b):
    return torch.where(a * b < 0, torch.zeros_like(a), torch.where(a.abs() < b.abs(), a, b))


def _recip4(x):
    y = x + 1.0e-12
    y = y * y
    return 1.0 / (y * y)


def _weno3_1d(m2, m1, z, p1, p2):
    s = [-2.0 * m1 + 0.5 * m2 + 1.5 * z, 0.5 * (p1 - m1), -1.5 * z + 2.0 * p1 - 0.5 * p2]
    c = [0.5 * (m2 - 2.0 * m1 + z), 0.5 * (m1 - 2.0 * z + p1), 0.5 * (z - 2.0 * p1 + p2)]
    wt = []
    for k in range(3):
        y = s[k] * s[k] + (13.0 / 3.0) * c[k] * c[k] + 1.0e-12
        y = y * y
        wt.append((100.0 if k == 1 else 1.0) / (y * y))
    total = wt[0] + wt[1] + wt[2]
    wt = [v / total for v in wt]
    return wt[0] * s[0] + wt[1] * s[1] + wt[2] * s[2], wt[0] * c[0] + wt[1] * c[1] + wt[2] * c[2]


def _coefficients(order, at):
    """Modal coefficients from at(dj, di), the field shifted by whole cells."""
    z, e, w, n, s = at(0, 0), at(0, 1), at(0, -1), at(1, 0), at(-1, 0)
    if order == 1:
        return [z, _minmod(e - z, z - w), _minmod(n - z, z - s)]
    ne, se, nw, sw = at(1, 1), at(-1, 1), at(1, -1), at(-1, -1)
    ee, ww, nn, ss = at(0, 2), at(0, -2), at(2, 0), at(-2, 0)
    if order == 2:
        c1, c3 = _weno3_1d(ww, w, z, e, ee)
        c2, c4 = _weno3_1d(ss, s, z, n, nn)
        xy = [ne - z - c1 - c2 - c3 - c4, -se + z + c1 - c2 + c3 + c4, -nw + z - c1 + c2 + c3 + c4, sw - z + c1 + c2 - c3 - c4]
        t = 4.0 * (c3 * c3 + c4 * c4)
        wt = [_recip4(t + v * v) for v in xy]
        total = wt[0] + wt[1] + wt[2] + wt[3]
        wt = [v / total for v in wt]
        return [z, c1, c2, c3, c4, wt[0] * xy[0] + wt[1] * xy[1] + wt[2] * xy[2] + wt[3] * xy[3]]
    # order 3: a fourth-degree central polynomial and five third-degree ones
    gam = 0.85
    top = [41.0 / 60.0 * (-w + e) + 11.0 / 120.0 * (ww - ee), 41.0 / 60.0 * (-s + n) + 11.0 / 120.0 * (ss - nn),
           -z + 0.5 * (w + e), -z + 0.5 * (s + n), 0.25 * (sw - nw - se + ne)]
    xxx, yyy = (w - e) / 6.0 + (ee - ww) / 12.0, (s - n) / 6.0 + (nn - ss) / 12.0
    xxy = 0.25 * (-sw + nw - se + ne) + 0.5 * (s - n)
    xyy = 0.5 * (w - e) + 0.25 * (ne - sw - nw + se)
    x, y, xx, yy, xy = top
    ind = ((x + 0.1 * xxx) ** 2 + 13.0 / 3.0 * (xx * xx + yy * yy) + (y + 0.1 * yyy) ** 2
           + 39.05 * (xxx * xxx + yyy * yyy) + 7.0 / 6.0 * xy * xy + 4.7 * (xxy * xxy + xyy * xyy))
    cx, cy, cxx, cyy = 0.5 * (e - w), 0.5 * (n - s), -z + 0.5 * (w + e), -z + 0.5 * (s + n)
    low = [
        [cx, cy, cxx, cyy, 0.25 * (sw - nw - se + ne)],
        [1.5 * z - 2.0 * w + 0.5 * ww, cy, 0.5 * z - w + 0.5 * ww, cyy, 0.5 * (sw - nw - s + n)],
        [-1.5 * z + 2.0 * e - 0.5 * ee, cy, 0.5 * z - e + 0.5 * ee, cyy, 0.5 * (-se + ne + s - n)],
        [cx, 1.5 * z - 2.0 * s + 0.5 * ss, cxx, 0.5 * z - s + 0.5 * ss, 0.5 * (-w + sw + e - se)],
        [cx, -1.5 * z + 2.0 * n - 0.5 * nn, cxx, 0.5 * z - n + 0.5 * nn, 0.5 * (w - nw - e + ne)],
    ]
    lin = [(1.0 - gam) * gam] + [0.25 * (1.0 - gam) * (1.0 - gam)] * 4
    wt4 = gam * _recip4(ind)
    wts = [lin[k] * _recip4(p[0] ** 2 + p[1] ** 2 + 13.0 / 3.0 * (p[2] ** 2 + p[3] ** 2) + 7.0 / 6.0 * p[4] ** 2)
           for k, p in enumerate(low)]
    total = wt4 + sum(wts)
    ratio = wt4 / total / gam
    wts = [v / total for v in wts]
    out = [z]
    for k in range(5):
        out.append(ratio * (top[k] - sum(lin[m] * low[m][k] for m in range(5))) + sum(wts[m] * low[m][k] for m in range(5)))
    return out + [ratio * xxx, ratio * yyy, ratio * xxy, ratio * xyy]


def _basis(x, y, n):
    a = 1.0 / 12.0
    return [1.0, x, y, x * x - a, y * y - a, x * y, x * (x * x - 0.15), y * (y * y - 0.15), y * (x * x - a), x * (y * y - a)][:n]


def _basis_grad(x, y, n):
    a = 1.0 / 12.0
    gx = [0.0, 1.0, 0.0, 2 * x, 0.0, y, 3 * x * x - 0.15, 0.0, 2 * x * y, y * y - a][:n]
    gy = [0.0, 0.0, 1.0, 0.0, 2 * y, x, 0.0, 3 * y * y - 0.15, x * x - a, 2 * x * y][:n]
    return gx, gy


def _combine(co, phi):
    out = None
    for c, f in zip(co, phi):
        if f != 0.0:
            out = c * f if out is None else out + c * f
    return out if out is not None else torch.zeros_like(co[0])


def _rhs(g, U):
    """(right-hand side, dt) of the state U, shape (ny, nx, nvar)."""
    nx, ny, nv, order = g["nx"], g["ny"], NVAR[g["system"]], g["order"]
    h = (g["domain"][1] - g["domain"][0]) / nx
    q = list(U.unbind(-1))
    planes = _ghosted(g, _to_prim(g, q) if g["prim"] else q)
    # coefficients of the grid and one ring around it
    ring = [(lambda dj, di, a=a: a[2 + dj:ny + 4 + dj, 2 + di:nx + 4 + di]) for a in planes]
    co = [_coefficients(order, at) for at in ring]
    n = len(co[0])
    gp = 0.28867513459481287
    pts = [0.0] if order == 1 else [-gp, gp]
    nodes = {"E": [(0.5, s) for s in pts], "W": [(-0.5, s) for s in pts], "N": [(s, 0.5) for s in pts], "S": [(s, -0.5) for s in pts]}
    ok = None
    for side in nodes.values():
        for x, y in side:
            good = _admissible(g, [_combine(c, _basis(x, y, n)) for c in co])
            ok = good if ok is None else ok & good
    for c, at in zip(co, ring):  # where the check fails: minmod slopes, or the mean alone
        z = at(0, 0)
        flat = [z, _minmod(at(0, 1) - z, z - at(0, -1)), _minmod(at(1, 0) - z, z - at(-1, 0))] if g["prim"] else [z]
        for k in range(n):
            c[k] = torch.where(ok, c[k], flat[k] if k < len(flat) else torch.zeros_like(z))
    # volume term
    res = [torch.zeros_like(q[0]) for _ in range(nv)]
    inner = [[a[1:-1, 1:-1] for a in c] for c in co]
    for x in pts:
        for y in pts:
            gx, gy = _basis_grad(x, y, n)
            B = _nonconservative(g, [_combine(c, _basis(x, y, n)) for c in inner], [_combine(c, gx) / h for c in inner],
                                 [_combine(c, gy) / h for c in inner])
            for c in range(nv):
                if B[c] is not None:
                    res[c] = res[c] - B[c] / len(pts) ** 2
    # faces
    smax = 0.0
    for axis, (lo, hi) in enumerate((("E", "W"), ("N", "S"))):
        for (xl, yl), (xr, yr) in zip(nodes[lo], nodes[hi]):
            left = [_combine(c, _basis(xl, yl, n)) for c in co]
            right = [_combine(c, _basis(xr, yr, n)) for c in co]
            if axis == 0:
                left, right = [a[1:-1, :-1] for a in left], [a[1:-1, 1:] for a in right]
            else:
                left, right = [a[:-1, 1:-1] for a in left], [a[1:, 1:-1] for a in right]
            fl, sl, ql = _flux(g, left, axis)
            fr, sr, qr = _flux(g, right, axis)
            s = torch.maximum(sl, sr)
            smax = max(smax, float(s.max()))
            jump = [b - a for a, b in zip(left, right)]
            none = [torch.zeros_like(s)] * nv
            D = _nonconservative(g, [0.5 * (a + b) for a, b in zip(left, right)], jump if axis == 0 else none, none if axis == 0 else jump)
            for c in range(nv):
                F = 0.5 * (fr[c] + fl[c] - s * (qr[c] - ql[c])) / len(pts)
                up, dn = (F[:, 1:], F[:, :-1]) if axis == 0 else (F[1:], F[:-1])
                res[c] = res[c] - (up - dn) / h
                if D[c] is not None:
                    up, dn = (D[c][:, 1:], D[c][:, :-1]) if axis == 0 else (D[c][1:], D[c][:-1])
                    res[c] = res[c] - 0.5 * (up + dn) / len(pts) / h
    return torch.stack(res, -1), (CFL * h) / (2.0 * smax)
