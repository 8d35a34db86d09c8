"""Performance cases: the calls a user of smilei_amd makes, over the range of
sizes, orders, precision forms and options the library is used with.

Three kinds of case:

* "sim"     -- the engine: a resident ``Simulation`` advanced some time steps
               between two diagnostics; one pass returns what the diagnostics
               read (the E, B and J fields, the charge density of all species
               and the energies);
* "patch"   -- the operators of one patch, as a host code with its own
               orchestration calls them (interpolator, pusher, projector), and
               "seam", the reference's own deposition entry points;
* "patches" -- the synchronisation between the patches of a device: J ghost
               sum, per-patch Yee solver, B exchange, particle exchange + sort.

``exact`` restates each of them in plain torch, in 64 bits.
"""
import ctypes
import math

import numpy as np
import torch

import smilei_amd as sa
from smilei_amd import _lib

DEV = "cuda"
F64 = torch.float64
FIELDS = ("Ex", "Ey", "Ez", "Bx", "By", "Bz", "Jx", "Jy", "Jz")


def listed():
    return [
        # the smallest whole simulation: launches and their latency (test-sized box, a diagnostic every 50 steps)
        dict(name="sim_mixed_small", kind="sim", form="mixed", order=2, nx=32, ny=32, nz=32, px=16, py=16, pz=16,
             plasma="thermal", ppc=8, sigma=0.05, steps=50, tuned=False),
        # the 67M-particle thermal plasma of bench.py, run as bench.py runs it
        dict(name="sim_mixed_thermal", kind="sim", form="mixed", order=2, nx=256, ny=128, nz=128, px=16, py=16, pz=16,
             plasma="resident", ppc=8, sigma=0.05, steps=50, tuned=True),
        # laser-wakefield-like box: uneven patches, half a particle per cell behind a ramp, relativistic quiver
        dict(name="sim_mixed_lwfa", kind="sim", form="mixed", order=2, nx=256, ny=64, nz=64, px=32, py=16, pz=16,
             plasma="lwfa", ppc=1, sigma=0.0, steps=20, tuned=True),
        # fourth-order shapes, mixed form
        dict(name="sim_mixed_o4", kind="sim", form="mixed", order=4, nx=64, ny=64, nz=64, px=16, py=16, pz=16,
             plasma="thermal", ppc=8, sigma=0.05, steps=10, tuned=False),
        # the drop-in FP64 form on a small beam-plasma (two backgrounds and a gamma = 50 beam)
        dict(name="sim_fp64_beam", kind="sim", form="fp64", order=2, nx=96, ny=64, nz=64, px=32, py=16, pz=16,
             plasma="beam", ppc=6, sigma=0.02, steps=10, tuned=False),
        # FP64, fourth order, 12-cell patches and an odd number of particles per cell
        dict(name="sim_fp64_o4", kind="sim", form="fp64", order=4, nx=48, ny=36, nz=48, px=12, py=12, pz=12,
             plasma="thermal", ppc=5, sigma=0.05, steps=10, tuned=False),
        # 2D3V plasma
        dict(name="sim_2d", kind="sim", form="fp64", order=2, nx=512, ny=512, nz=1, px=32, py=32, pz=1,
             plasma="thermal", ppc=16, sigma=0.05, steps=20, tuned=False),
        # the reproducible deposit (summation order of the reference)
        dict(name="sim_deterministic", kind="sim", form="det", order=2, nx=32, ny=32, nz=32, px=8, py=8, pz=8,
             plasma="thermal", ppc=8, sigma=0.05, steps=2, tuned=False),
        # one small patch of a host code's own loop: interpolate, push, project
        dict(name="patch_o2_small", kind="patch", order=2, nx=16, ny=16, nz=16, ppc=8, sigma=0.05),
        # one large patch, fourth order
        dict(name="patch_o4_large", kind="patch", order=4, nx=64, ny=64, nz=64, ppc=8, sigma=0.05),
        # the reference's device projector: binned particles, currents and density
        dict(name="seam_deposit", kind="seam", order=2, nx=32, ny=32, nz=32, ppc=16, sigma=0.1),
        # everything between the patches of one device for one step
        dict(name="patches_exchange", kind="patches", order=2, nx=64, ny=64, nz=64, px=32, py=32, pz=32, ppc=16,
             sigma=0.1),
    ]


def _log(rng, lo, hi):
    return math.exp(rng.uniform(math.log(lo), math.log(hi)))


def draw(rng):
    kind = rng.choice(["sim", "sim", "sim", "sim", "patch", "patch", "seam", "patches"])
    if kind == "sim":
        form, order, nd = rng.choice([("mixed", 2, 3), ("mixed", 2, 3), ("mixed", 4, 3), ("fp64", 2, 3), ("fp64", 4, 3),
                                      ("fp64", 2, 2), ("det", 2, 3)])
        patch = [rng.choice([12, 16, 24, 32] if order == 4 else [8, 12, 16, 20, 32]) for _ in range(3)]
        top = 1.5e5 if form == "det" else (6e5 if order == 4 else 2.5e6)  # cells x particles per cell
        total = _log(rng, 4e4, top)
        ppc = rng.choice([1, 2, 3, 4, 5, 7, 8, 11, 16])
        side = max(8.0, (total / ppc) ** (1.0 / nd))
        n = [max(1, round(side * rng.uniform(0.7, 1.4) / p)) * p for p in patch]
        if nd == 2:
            n[2] = patch[2] = 1
        plasma = rng.choice(["thermal", "thermal", "beam"] if nd == 3 else ["thermal"])
        return dict(kind="sim", form=form, order=order, nx=n[0], ny=n[1], nz=n[2], px=patch[0], py=patch[1],
                    pz=patch[2], plasma=plasma, ppc=ppc, sigma=rng.choice([0.01, 0.02, 0.05, 0.1]),
                    steps=rng.choice([2, 3]) if form == "det" else rng.choice([5, 10, 20]), tuned=False)
    if kind == "patch" or kind == "seam":
        order = rng.choice([2, 4]) if kind == "patch" else 2
        n = [round(_log(rng, 12, 56)) for _ in range(3)]
        if kind == "seam":  # whole 4^3 bins
            n = [max(12, v // 4 * 4) for v in n]
        return dict(kind=kind, order=order, nx=n[0], ny=n[1], nz=n[2], ppc=rng.choice([1, 3, 5, 8, 13]),
                    sigma=rng.choice([0.02, 0.05, 0.1, 0.5]))
    p = [rng.choice([8, 12, 16, 32]) for _ in range(3)]
    n = [p[d] * max(1, round(_log(rng, 16, 56) / p[d])) for d in range(3)]
    return dict(kind="patches", order=2, nx=n[0], ny=n[1], nz=n[2], px=p[0], py=p[1], pz=p[2],
                ppc=rng.choice([1, 3, 5, 8, 16]), sigma=rng.choice([0.02, 0.1, 0.5]))


# ---------------------------------------------------------------------------
# Inputs
# ---------------------------------------------------------------------------
def _generator(seed):
    g = torch.Generator(device=DEV)
    g.manual_seed(seed)
    return g


def _cells_dx(case):
    """Cells and cell lengths of the axes of the case (two in 2D)."""
    n = [case["nx"], case["ny"], case["nz"]]
    if case["nz"] == 1:
        return n[:2], [0.2, 0.2]
    return n, {"lwfa": [0.1, 0.5, 0.5], "beam": [0.25] * 3}.get(case.get("plasma"), [0.2] * 3)


def _timestep(dx):
    return 0.95 / math.sqrt(sum(1.0 / d ** 2 for d in dx))


def _uniform(g, n, dx, cells, ppc):
    """ppc particles at random positions of each of the given cells."""
    t = cells.repeat_interleave(ppc)
    strides = [math.prod(n[d + 1:]) for d in range(len(n))]
    pos = []
    for d in range(len(n)):
        i = (t // strides[d]) % n[d]
        v = (i + torch.rand(len(t), generator=g, device=DEV, dtype=F64)) * dx[d]
        pos.append(torch.clamp(v, max=math.nextafter(n[d] * dx[d], 0.0)))
    return pos


def _particles(g, n, dx, cells, ppc, sigma, density=1.0, drift=0.0):
    pos = _uniform(g, n, dx, cells, ppc)
    m = len(pos[0])
    u = sigma * torch.randn(3, m, generator=g, device=DEV, dtype=F64)
    u[0] += drift
    w = torch.full((m,), density * math.prod(dx) / ppc, device=DEV, dtype=F64)
    return pos, [u[0], u[1], u[2]], w


def _plasma(case, seed):
    """Species (name, mass, charge, positions, momenta, weights) and the
    initial fields of a sim case."""
    g = _generator(seed)
    n, dx = _cells_dx(case)
    every = torch.arange(math.prod(n), device=DEV)
    kind, ppc, s = case["plasma"], case["ppc"], case["sigma"]
    if kind == "lwfa":
        idx = [(every // (n[1] * n[2])), (every // n[2]) % n[1], every % n[2]]
        c = [(idx[d] + 0.5) * dx[d] for d in range(3)]
        r2 = (c[1] - 0.5 * n[1] * dx[1]) ** 2 + (c[2] - 0.5 * n[2] * dx[2]) ** 2
        dens = 0.01 * torch.clamp((c[0] - n[0] / 8 * dx[0]) / (n[0] / 5 * dx[0]), 0.0, 1.0) * (1 + 0.5 * r2 / 400.0)
        cells = every[((idx[0] + idx[1] + idx[2]) % 2 == 0) & (dens > 0)]
        pos, u, _ = _particles(g, n, dx, cells, ppc, s)
        w = dens[cells].repeat_interleave(ppc) * math.prod(dx) / ppc
        x, y, z = torch.meshgrid(*[torch.arange(n[d], device=DEV, dtype=F64) * dx[d] for d in range(3)], indexing="ij")
        r2 = (y - 0.5 * n[1] * dx[1]) ** 2 + (z - 0.5 * n[2] * dx[2]) ** 2
        xl = n[0] * dx[0] / 3
        laser = 2.0 * torch.exp(-r2 / 64.0 - (x - xl) ** 2 / 9.0) * torch.sin(x - xl)
        return [("electron", 1.0, -1.0, pos, u, w)], {"Ey": laser, "Bz": laser}
    sp = [("electron", 1.0, -1.0) + _particles(g, n, dx, every, ppc, s),
          ("proton", 1836.0, 1.0) + _particles(g, n, dx, every, ppc, s / math.sqrt(1836.0))]
    if kind == "beam":
        ry, rz = (every // n[2]) % n[1] + 0.5 - 0.5 * n[1], every % n[2] + 0.5 - 0.5 * n[2]
        cells = every[ry * ry + rz * rz <= (min(n[1], n[2]) / 4) ** 2]
        sp.append(("beam", 1.0, -1.0) + _particles(g, n, dx, cells, 8, 0.0, 0.1, math.sqrt(2499.0)))
    return sp, {}


def _ptr(t):
    return ctypes.c_void_p(t.data_ptr())


def _ints(v):
    return (ctypes.c_int * 3)(*[int(a) for a in v])


def _doubles(v):
    return (ctypes.c_double * 3)(*[float(a) for a in v])


#: staggering (1 = dual) of the components along x, y, z
DUAL = {"Ex": (1, 0, 0), "Ey": (0, 1, 0), "Ez": (0, 0, 1), "Bx": (0, 1, 1), "By": (1, 0, 1), "Bz": (1, 1, 0),
        "Jx": (1, 0, 0), "Jy": (0, 1, 0), "Jz": (0, 0, 1)}


def _patch_shape(name, n, order):
    return tuple(n[d] + 2 * order + 1 + DUAL[name][d] for d in range(3))


def _patch_fields(g, n, order, scale=0.05):
    return {f: scale * torch.randn(_patch_shape(f, n, order), generator=g, device=DEV, dtype=F64)
            for f in ("Ex", "Ey", "Ez", "Bx", "By", "Bz")}


def _patch_inputs(case, seed):
    g = _generator(seed)
    n, dx = _cells_dx(case)
    pos, u, w = _particles(g, n, dx, torch.arange(math.prod(n), device=DEV), case["ppc"], case["sigma"])
    return dict(n=n, dx=dx, dt=_timestep(dx), x=pos, u=u, w=w, F=_patch_fields(g, n, case["order"]))


def _seam_inputs(case, seed):
    """Particles of one patch in 4^3 bins (x-major), the interpolator's old
    nodes and offsets, and their positions after a push."""
    g = _generator(seed)
    n, dx = _cells_dx(case)
    dt = _timestep(dx)
    t = torch.arange(math.prod(n), device=DEV)
    c = [t // (n[1] * n[2]), (t // n[2]) % n[1], t % n[2]]
    nb = [v // 4 for v in n]
    bins = ((c[0] // 4) * nb[1] + c[1] // 4) * nb[2] + c[2] // 4
    cells = t[torch.argsort(bins, stable=True)]
    pos, u, w = _particles(g, n, dx, cells, case["ppc"], case["sigma"])
    w *= 0.5 + torch.rand(len(w), generator=g, device=DEV, dtype=F64)
    charge = torch.randint(1, 4, (len(w),), generator=g, device=DEV).to(torch.int16)
    pn = [pos[d] / dx[d] for d in range(3)]
    node = [torch.round(v) for v in pn]
    gam = torch.sqrt(1.0 + u[0] ** 2 + u[1] ** 2 + u[2] ** 2)
    return dict(n=n, dx=dx, dt=dt, nb=nb, w=w, charge=charge, new=[pos[d] + dt * u[d] / gam for d in range(3)],
                iold=torch.stack([node[d] + case["order"] for d in range(3)]).to(torch.int32),
                delta=torch.stack([pn[d] - node[d] for d in range(3)]), invgf=1.0 / gam,
                ends=torch.arange(1, math.prod(nb) + 1, device=DEV, dtype=torch.int32) * (64 * case["ppc"]))


def _patches_inputs(case, seed):
    g = _generator(seed)
    n, dx = _cells_dx(case)
    patch = [case["px"], case["py"], case["pz"]]
    npatch = [n[d] // patch[d] for d in range(3)]
    count = math.prod(npatch)

    def stack(names):
        return torch.cat([0.05 * torch.randn((count, math.prod(_patch_shape(f, patch, case["order"]))), generator=g,
                                             device=DEV, dtype=F64) for f in names], 1)

    pos, u, w = _particles(g, n, dx, torch.arange(math.prod(n), device=DEV), case["ppc"], case["sigma"])
    charge = torch.randint(1, 4, (len(w),), generator=g, device=DEV).to(torch.int16)
    return dict(n=n, dx=dx, dt=_timestep(dx), patch=patch, npatch=npatch, x=pos, u=u, w=w, charge=charge,
                J=stack(("Jx", "Jy", "Jz")), E=stack(("Ex", "Ey", "Ez")), B=stack(("Bx", "By", "Bz")))


# ---------------------------------------------------------------------------
# The cases
# ---------------------------------------------------------------------------
def prepare(case, seed):
    return {"sim": _prepare_sim, "patch": _prepare_patch, "seam": _prepare_seam,
            "patches": _prepare_patches}[case["kind"]](case, seed)


def run(state):
    return state["run"](state)


def _prepare_sim(case, seed):
    n, dx = _cells_dx(case)
    nd = len(n)
    sim = sa.Simulation("3Dcartesian" if nd == 3 else "2Dcartesian", case["order"], n,
                        [case["px"], case["py"], case["pz"]][:nd], dx, _timestep(dx),
                        precision=sa.MIXED if case["form"] == "mixed" else sa.PLAIN_FP64,
                        deposit=sa.DEPOSIT_DETERMINISTIC if case["form"] == "det" else sa.DEPOSIT_ATOMIC)
    if case["plasma"] == "resident":
        for name, mass, q in (("electron", 1.0, -1.0), ("proton", 1836.0, 1.0)):
            sid = sim.add_species(name, mass, q, math.prod(n) * case["ppc"])
            sim.init_species(sid, case["ppc"], 1.0, case["sigma"] / math.sqrt(mass), seed=seed)
    else:
        species, fields = _plasma(case, seed)
        for name, mass, q, pos, u, w in species:
            sid = sim.add_species(name, mass, q, len(w))
            z = pos[2] if nd == 3 else torch.zeros_like(w)
            sim.set_particles(sid, *[t.cpu().numpy() for t in (pos[0], pos[1], z, u[0], u[1], u[2], w)])
        for name, f in fields.items():
            sim.set_field(name, f.cpu().numpy())
            if name[0] == "B":
                sim.set_field(name + "_m", f.cpu().numpy())
    if case["tuned"]:  # the order inside a cell left to the scatter, the launch shapes to the autotuner (bench.py)
        sim.set_tuning(sa.TUNE_CELL_ORDER, 0)
        sim.autotune()
    return dict(run=_run_sim, sim=sim, steps=case["steps"])


def _run_sim(s):
    s["sim"].step(s["steps"])
    out = {f: s["sim"].get_field(f) for f in FIELDS}
    out["rho"] = s["sim"].rho()
    out["energies"] = s["sim"].energies()
    return out


def _prepare_patch(case, seed):
    s = _patch_inputs(case, seed)
    m = len(s["w"])
    shapes = [_patch_shape(f, s["n"], case["order"]) for f in ("Jx", "Jy", "Jz")]
    s["jbuf"] = torch.zeros(sum(map(math.prod, shapes)), device=DEV, dtype=F64)
    s["J"] = [t.view(shapes[c]) for c, t in enumerate(s["jbuf"].split([math.prod(v) for v in shapes]))]
    s["Ep"], s["Bp"], s["delta"] = (torch.zeros(3, m, device=DEV, dtype=F64) for _ in range(3))
    s["iold"] = torch.zeros(3, m, device=DEV, dtype=torch.int32)
    s["invgf"] = torch.zeros(m, device=DEV, dtype=F64)
    s.update(run=_run_patch, L=_lib.load(), order=case["order"])
    return s


def _run_patch(s):
    """One step of a single periodic patch in given fields."""
    L, order, n, dx, m = s["L"], s["order"], s["n"], s["dx"], len(s["w"])
    st = ctypes.c_void_p(torch.cuda.current_stream().cuda_stream)
    size, begin, length = _ints(v + 2 * order + 1 for v in n), _ints([-order] * 3), _doubles(dx)
    fields = [_ptr(s["F"][f]) for f in ("Ex", "Ey", "Ez", "Bx", "By", "Bz")]
    x, u = [_ptr(t) for t in s["x"]], [_ptr(t) for t in s["u"]]
    _lib.check(L.smi_interpolate_3d(order, *fields, size, begin, length, m, *x, _ptr(s["Ep"]), _ptr(s["Bp"]),
                                    _ptr(s["iold"]), _ptr(s["delta"]), st))
    _lib.check(L.smi_push_boris(3, -1.0, 1.0, s["dt"], m, *x, *u, _ptr(s["Ep"]), _ptr(s["Bp"]), _ptr(s["invgf"]), st))
    s["jbuf"].zero_()
    _lib.check(L.smi_currents_3d(order, *[_ptr(t) for t in s["J"]], size, begin, length, s["dt"], -1.0, m, *x,
                                 _ptr(s["w"]), _ptr(s["iold"]), _ptr(s["delta"]), 0, st))
    for d in range(3):
        s["x"][d].remainder_(n[d] * dx[d])
    return {"J": s["J"], "x": s["x"], "u": s["u"], "Ep": s["Ep"], "Bp": s["Bp"], "iold": s["iold"],
            "delta": s["delta"], "invgf": s["invgf"]}


def _prepare_seam(case, seed):
    s = _seam_inputs(case, seed)
    sizes = [math.prod(_patch_shape(f, s["n"], 2)) for f in ("Jx", "Jy", "Jz")] + [math.prod(v + 5 for v in s["n"])]
    s["buf"] = torch.zeros(sum(sizes), device=DEV, dtype=F64)
    s["out"] = list(s["buf"].split(sizes))
    s.update(run=_run_seam, L=_lib.load())
    return s


def _run_seam(s):
    L, dx, dt = s["L"], s["dx"], s["dt"]
    s["buf"].zero_()
    torch.cuda.current_stream().synchronize()  # the seams work on the null stream
    J, rho = s["out"][:3], s["out"][3]
    tail = ([_ptr(t) for t in s["new"]] + [_ptr(s["charge"]), _ptr(s["w"]), _ptr(s["ends"])] + s["nb"]
            + [_ptr(s["invgf"]), _ptr(s["iold"]), _ptr(s["delta"]), len(s["w"]), 1.0 / math.prod(dx)]
            + [1.0 / v for v in dx] + [v / dt for v in dx] + [-2, -2, -2, s["n"][1] + 5, s["n"][2] + 5, 1, True])
    _lib.check(L.smi_current_deposition_3d(*[_ptr(t) for t in J], *[t.numel() for t in J], *tail))
    _lib.check(L.smi_density_deposition_3d(_ptr(rho), rho.numel(), *tail))
    return {"J": J, "rho": rho}


def _prepare_patches(case, seed):
    s = _patches_inputs(case, seed)
    m, patches = len(s["w"]), math.prod(s["npatch"])
    s["fresh"], s["J"] = s["J"], torch.empty_like(s["J"])
    s["zero"], s["invgf"] = torch.zeros(3, m, device=DEV, dtype=F64), torch.zeros(m, device=DEV, dtype=F64)
    s["key"] = torch.zeros(m, device=DEV, dtype=torch.int32)
    s["count"] = torch.zeros(patches, device=DEV, dtype=torch.int32)
    s["ends"] = torch.zeros(patches * math.prod(v // 4 for v in s["patch"]), device=DEV, dtype=torch.int32)
    s["dims"] = [[_patch_shape(f, s["patch"], case["order"]) for f in names]
                 for names in (("Ex", "Ey", "Ez"), ("Bx", "By", "Bz"), ("Jx", "Jy", "Jz"))]
    s.update(run=_run_patches, L=_lib.load(), order=case["order"])
    return s


def _run_patches(s):
    """The synchronisation half of a step over all patches of a device."""
    L, order, m = s["L"], s["order"], len(s["w"])
    st = ctypes.c_void_p(torch.cuda.current_stream().cuda_stream)
    n, patch, length = _ints(s["n"]), _ints(s["patch"]), _doubles(s["dx"])
    size = _ints(v + 2 * order + 1 for v in s["patch"])
    s["J"].copy_(s["fresh"])  # the step's per-patch deposits
    _lib.check(L.smi_sum_j_ghosts(3, order, n, patch, _ptr(s["J"]), st))
    for p in range(math.prod(s["npatch"])):
        comp = []
        for a, dims in zip((s["E"], s["B"], s["J"]), s["dims"]):
            at = a.data_ptr() + 8 * p * a.shape[1]
            for d in dims:
                comp.append(ctypes.c_void_p(at))
                at += 8 * math.prod(d)
        _lib.check(L.smi_maxwell_ampere_3d(*comp, size, s["dt"], length, st))
        _lib.check(L.smi_maxwell_faraday_3d(*comp[3:6], *comp[:3], size, s["dt"], length, st))
    _lib.check(L.smi_exchange_b(3, order, n, patch, _ptr(s["B"]), st))
    x, u = [_ptr(t) for t in s["x"]], [_ptr(t) for t in s["u"]]
    _lib.check(L.smi_push_boris(3, -1.0, 1.0, s["dt"], m, *x, *u, _ptr(s["zero"]), _ptr(s["zero"]), _ptr(s["invgf"]),
                                st))
    _lib.check(L.smi_sort_exchange(3, n, patch, length, m, *x, *u, _ptr(s["w"]), _ptr(s["charge"]), _ptr(s["key"]),
                                   _ptr(s["count"]), _ptr(s["ends"]), st))
    return {"J": s["J"], "E": s["E"], "B": s["B"], "x": s["x"], "u": s["u"], "w": s["w"], "charge": s["charge"],
            "key": s["key"], "count": s["count"], "ends": s["ends"]}


# ---------------------------------------------------------------------------
# Work of one pass: inputs read once, outputs written once
# ---------------------------------------------------------------------------
def work(case):
    n, dx = _cells_dx(case)
    cells, order, nd = math.prod(n), case["order"], len(n)
    push = {(2, 2): 500.0, (3, 2): 1500.0, (3, 4): 6500.0}[(nd, order)]  # gather + Boris + Esirkepov, operations
    if case["kind"] == "sim":
        parts = cells * case["ppc"] * 2
        if case["plasma"] == "beam":
            parts = int(parts + cells * 8 * math.pi / 16)
        elif case["plasma"] == "lwfa":
            parts = int(cells * case["ppc"] * 0.5 * 7 / 8)
        per = 60 if case["form"] == "mixed" else (108 if nd == 3 else 92)
        # per cell and step: E, B, B_m in, E, B, B_m, J out
        return {"bytes": case["steps"] * (per * parts + 168 * cells) + 80 * cells + (per / 4) * parts,
                "flops": case["steps"] * (push * parts + 60 * cells)}
    parts = cells * case["ppc"]
    if case["kind"] == "patch":
        return {"bytes": parts * (48 + 8 + 48 + 48 + 12 + 24 + 8) + cells * 72, "flops": push * parts}
    if case["kind"] == "seam":
        return {"bytes": parts * 2 * (24 + 2 + 8 + 12 + 24) + cells * 32, "flops": 1400.0 * parts}
    slots = math.prod(n[d] // p for d, p in enumerate((case["px"], case["py"], case["pz"])))
    points = slots * math.prod(p + 5 for p in (case["px"], case["py"], case["pz"]))
    return {"bytes": parts * (2 * 7 * 8 + 2 * 2 + 4 + 8) + points * 8 * 15, "flops": 60.0 * points + 40.0 * parts}


# ---------------------------------------------------------------------------
# The same in plain torch, 64 bits
# ---------------------------------------------------------------------------
def _spline(order, d):
    if order == 2:
        return [0.5 * (d - 0.5) ** 2, 0.75 - d * d, 0.5 * (d + 0.5) ** 2]
    d2, d3, d4 = d ** 2, d ** 3, d ** 4
    return [1 / 384 - d / 48 + d2 / 16 - d3 / 12 + d4 / 24, 19 / 96 - 11 * d / 24 + d2 / 4 + d3 / 6 - d4 / 6,
            115 / 192 - 5 * d2 / 8 + d4 / 4, 19 / 96 + 11 * d / 24 + d2 / 4 - d3 / 6 - d4 / 6,
            1 / 384 + d / 48 + d2 / 16 + d3 / 12 + d4 / 24]


def _at(idx, dims, wrap):
    """Flat index of a grid point per particle (periodic if wrap)."""
    t = None
    for i, m in zip(idx, dims):
        i = torch.remainder(i, m) if wrap else i
        t = i if t is None else t * m + i
    return t


def _gather(field, dual, pn, order, begin, wrap):
    nd, H = len(pn), order // 2
    node, weight = [], []
    for d in range(nd):
        i = torch.round(pn[d] + 0.5 * dual[d])
        node.append(i.long() - begin[d])
        weight.append(_spline(order, pn[d] - i + 0.5 * dual[d]))
    flat, out = field.reshape(-1), torch.zeros_like(pn[0])
    dims = field.shape[:nd]
    for a in range(-H, H + 1):
        for b in range(-H, H + 1):
            for c in range(-H, H + 1) if nd == 3 else (None,):
                off = (a, b) if nd == 2 else (a, b, c)
                v = flat[_at([node[d] + off[d] for d in range(nd)], dims, wrap)]
                for d in range(nd):
                    v = v * weight[d][off[d] + H]
                out += v
    return out


def _boris(q_m, dt, E, B, u):
    a = [0.5 * dt * q_m * e for e in E]
    m = [u[d] + a[d] for d in range(3)]
    f = 0.5 * dt * q_m / torch.sqrt(1 + m[0] ** 2 + m[1] ** 2 + m[2] ** 2)
    t = [f * b for b in B]
    s = 2 / (1 + t[0] ** 2 + t[1] ** 2 + t[2] ** 2)

    def cross(p, r):
        return [p[1] * r[2] - p[2] * r[1], p[2] * r[0] - p[0] * r[2], p[0] * r[1] - p[1] * r[0]]

    c = cross(m, t)
    c = cross([m[d] + c[d] for d in range(3)], t)
    new = [m[d] + s * c[d] + a[d] for d in range(3)]
    return new, 1 / torch.sqrt(1 + new[0] ** 2 + new[1] ** 2 + new[2] ** 2)


def _shapes(order, old, new, node):
    """Old and new shape on the order + 3 points around the old node."""
    S = order + 3
    s0, s1 = torch.zeros(S, len(new), device=DEV, dtype=F64), torch.zeros(S, len(new), device=DEV, dtype=F64)
    for m, v in enumerate(_spline(order, old)):
        s0[m + 1] = v
    i = torch.round(new)
    sh = (i - node).long()
    for m, v in enumerate(_spline(order, new - i)):
        s1.scatter_(0, (sh + 1 + m).unsqueeze(0), v.unsqueeze(0))
    return s0, s1


def _deposit(J, order, delta, new, node, begin, cr, crz, wrap):
    """Esirkepov currents of the particles, added to J; node: old nearest
    node (global), new: new position in cells, cr: charge weight * dx / dt."""
    nd, S = len(new), order + 3
    sh = [_shapes(order, delta[d], new[d], node[d]) for d in range(nd)]
    s0, ds = [v[0] for v in sh], [v[1] - v[0] for v in sh]
    base = [node[d].long() - begin[d] - order // 2 - 1 for d in range(nd)]
    for c in range(nd):
        b, e = (c + 1) % nd, (c + 2) % nd
        dims, flat = J[c].shape[:nd], J[c].reshape(-1)
        for i in range(S):
            for j in range(S if nd == 3 else 1):
                if nd == 3:
                    wt = (s0[b][i] * s0[e][j] + 0.5 * ds[b][i] * s0[e][j] + 0.5 * s0[b][i] * ds[e][j]
                          + ds[b][i] * ds[e][j] / 3)
                else:
                    wt = s0[b][i] + 0.5 * ds[b][i]
                acc = torch.zeros_like(wt)
                for r in range(1, S):
                    acc = acc - cr[c] * ds[c][r - 1] * wt
                    off = {c: r, b: i}
                    if nd == 3:
                        off[e] = j
                    flat.index_add_(0, _at([base[d] + off[d] for d in range(nd)], dims, wrap), acc)
    if nd == 2:
        dims, flat = J[2].shape[:2], J[2].reshape(-1)
        for i in range(S):
            for j in range(S):
                a0, a1, b0, b1 = s0[0][i], s0[0][i] + ds[0][i], s0[1][j], s0[1][j] + ds[1][j]
                v = crz * (b0 * (0.5 * a1 + a0) + b1 * (0.5 * a0 + a1))
                flat.index_add_(0, _at([base[0] + i, base[1] + j], dims, wrap), v)


def _density(rho, order, pn, begin, cw, wrap):
    """Charge density of particles at pn (in cells), added to rho."""
    nd, H = len(pn), order // 2
    node = [torch.round(v) for v in pn]
    S = [_spline(order, pn[d] - node[d]) for d in range(nd)]
    dims, flat = rho.shape[:nd], rho.reshape(-1)
    for a in range(-H, H + 1):
        for b in range(-H, H + 1):
            for c in range(-H, H + 1) if nd == 3 else (None,):
                off = (a, b) if nd == 2 else (a, b, c)
                v = cw
                for d in range(nd):
                    v = v * S[d][off[d] + H]
                flat.index_add_(0, _at([node[d].long() - begin[d] + off[d] for d in range(nd)], dims, wrap), v)


def _exact_sim(case, seed):
    n, dx = _cells_dx(case)
    nd, order, dt = len(n), case["order"], _timestep(dx)
    species, init = _plasma(case, seed)
    shape = tuple(n) if nd == 3 else (n[0], n[1], 1)
    F = {f: torch.zeros(shape, device=DEV, dtype=F64) for f in FIELDS}
    for k, v in init.items():
        F[k] = v.clone()
    Bm = [F["Bx"].clone(), F["By"].clone(), F["Bz"].clone()]
    vol = math.prod(dx)

    def up(f, d):
        return torch.roll(f, -1, d) - f if d < nd else torch.zeros_like(f)

    def down(f, d):
        return f - torch.roll(f, 1, d) if d < nd else torch.zeros_like(f)

    k = [dt / dx[d] if d < nd else 0.0 for d in range(3)]
    for _ in range(case["steps"]):
        J = [torch.zeros(shape, device=DEV, dtype=F64) for _ in range(3)]
        moved = []
        for name, mass, q, pos, u, w in species:
            pn = [pos[d] / dx[d] for d in range(nd)]
            E = [_gather(F[f], DUAL[f], pn, order, [0] * nd, True) for f in ("Ex", "Ey", "Ez")]
            B = [_gather(Bm[c], DUAL[f], pn, order, [0] * nd, True) for c, f in enumerate(("Bx", "By", "Bz"))]
            un, invg = _boris(q / mass, dt, E, B, u)
            new = [pos[d] + dt * un[d] * invg for d in range(nd)]
            node = [torch.round(v) for v in pn]
            cw = q * w / vol
            _deposit(J, order, [pn[d] - node[d] for d in range(nd)], [new[d] / dx[d] for d in range(nd)], node,
                     [0] * nd, [cw * dx[d] / dt for d in range(nd)], cw * un[2] * invg / 3, True)
            moved.append((name, mass, q, [torch.remainder(new[d], n[d] * dx[d]) for d in range(nd)], un, w))
        species = moved
        F["Jx"], F["Jy"], F["Jz"] = J
        F["Ex"] = F["Ex"] - dt * J[0] + k[1] * up(F["Bz"], 1) - k[2] * up(F["By"], 2)
        F["Ey"] = F["Ey"] - dt * J[1] - k[0] * up(F["Bz"], 0) + k[2] * up(F["Bx"], 2)
        F["Ez"] = F["Ez"] - dt * J[2] + k[0] * up(F["By"], 0) - k[1] * up(F["Bx"], 1)
        new = [F["Bx"] - k[1] * down(F["Ez"], 1) + k[2] * down(F["Ey"], 2),
               F["By"] - k[2] * down(F["Ex"], 2) + k[0] * down(F["Ez"], 0),
               F["Bz"] - k[0] * down(F["Ey"], 0) + k[1] * down(F["Ex"], 1)]
        Bm = [(new[c] + F[f]) * 0.5 for c, f in enumerate(("Bx", "By", "Bz"))]
        F["Bx"], F["By"], F["Bz"] = new
    energies = [0.0]
    for f, comp in (("Ex", F["Ex"]), ("Ey", F["Ey"]), ("Ez", F["Ez"]), ("Bx", Bm[0]), ("By", Bm[1]), ("Bz", Bm[2])):
        sq = comp ** 2  # points of the periodic images count again (Field3D::norm2 over every patch's own points)
        for d in range(nd):
            m = torch.ones(n[d], device=DEV, dtype=F64)
            m[0] = 2
            if DUAL[f][d]:
                m[1] = 2
            sq = sq * m.view([-1 if e == d else 1 for e in range(3)])
        energies[0] += 0.5 * vol * float(sq.sum())
    for name, mass, q, pos, u, w in species:
        u2 = u[0] ** 2 + u[1] ** 2 + u[2] ** 2
        energies.append(mass * float((w * u2 / (1 + torch.sqrt(1 + u2))).sum()))
    F["rho"] = torch.zeros(shape, device=DEV, dtype=F64)
    for name, mass, q, pos, u, w in species:
        _density(F["rho"], order, [pos[d] / dx[d] for d in range(nd)], [0] * nd, q * w / vol, True)
    out = {f: v.cpu().numpy() for f, v in F.items()}
    out["energies"] = np.array(energies)
    return out


def _exact_patch(case, seed):
    s = _patch_inputs(case, seed)
    order, n, dx, dt = case["order"], s["n"], s["dx"], s["dt"]
    begin = [-order] * 3
    pn = [s["x"][d] / dx[d] for d in range(3)]
    E = [_gather(s["F"][f], DUAL[f], pn, order, begin, False) for f in ("Ex", "Ey", "Ez")]
    B = [_gather(s["F"][f], DUAL[f], pn, order, begin, False) for f in ("Bx", "By", "Bz")]
    u, invg = _boris(-1.0, dt, E, B, s["u"])
    new = [s["x"][d] + dt * u[d] * invg for d in range(3)]
    node = [torch.round(v) for v in pn]
    J = [torch.zeros(_patch_shape(f, n, order), device=DEV, dtype=F64) for f in ("Jx", "Jy", "Jz")]
    cw = -s["w"] / math.prod(dx)
    delta = [pn[d] - node[d] for d in range(3)]
    _deposit(J, order, delta, [new[d] / dx[d] for d in range(3)], node, begin, [cw * dx[d] / dt for d in range(3)],
             None, False)
    return {"J": J, "x": [torch.remainder(new[d], n[d] * dx[d]) for d in range(3)], "u": u, "Ep": torch.stack(E),
            "Bp": torch.stack(B), "iold": None, "delta": torch.stack(delta), "invgf": invg}


def _exact_seam(case, seed):
    s = _seam_inputs(case, seed)
    n, dx, dt = s["n"], s["dx"], s["dt"]
    begin = [-2] * 3
    node = [s["iold"][d].to(F64) - 2 for d in range(3)]
    new = [s["new"][d] / dx[d] for d in range(3)]
    cw = s["charge"].to(F64) * s["w"] / math.prod(dx)
    J = [torch.zeros(_patch_shape(f, n, 2), device=DEV, dtype=F64) for f in ("Jx", "Jy", "Jz")]
    _deposit(J, 2, s["delta"], new, node, begin, [cw * dx[d] / dt for d in range(3)], None, False)
    rho = torch.zeros([v + 5 for v in n], device=DEV, dtype=F64)
    _density(rho, 2, new, begin, cw, False)
    return {"J": [t.reshape(-1) for t in J], "rho": rho.reshape(-1)}


def _exact_patches(case, seed):
    s = _patches_inputs(case, seed)
    n, dx, dt, patch, npatch, os_ = s["n"], s["dx"], s["dt"], s["patch"], s["npatch"], case["order"]

    def views(a, names):
        out, at = [], 0
        for f in names:
            sh = _patch_shape(f, patch, os_)
            out.append(a[:, at:at + math.prod(sh)].clone().view(npatch + list(sh)))
            at += math.prod(sh)
        return out

    def cut(f, d, lo, hi):
        return f.narrow(3 + d, lo, hi - lo)

    def flat(v):
        return torch.cat([f.reshape(math.prod(npatch), -1) for f in v], 1)

    names = [("Ex", "Ey", "Ez"), ("Bx", "By", "Bz"), ("Jx", "Jy", "Jz")]
    E, B, J = (views(s[k], v) for k, v in zip("EBJ", names))
    for d in range(3):
        for c in range(3):  # overlap of the low neighbour's last and this patch's first planes
            g = 2 * os_ + 1 + (c == d)
            low = torch.roll(J[c], 1, d)
            tot = cut(low, d, patch[d], patch[d] + g) + cut(J[c], d, 0, g)
            cut(J[c], d, patch[d], patch[d] + g).copy_(torch.roll(tot, -1, d))
            cut(J[c], d, 0, g).copy_(tot)
    k = [dt / v for v in dx]

    def diff(f, d):
        return torch.diff(f, dim=3 + d)

    for c in range(3):
        b, e = (c + 1) % 3, (c + 2) % 3
        E[c] += -dt * J[c] + k[b] * diff(B[e], b) - k[e] * diff(B[b], e)
    for c in range(3):
        b, e = (c + 1) % 3, (c + 2) % 3
        inner = cut(cut(B[c], b, 1, B[c].shape[3 + b] - 1), e, 1, B[c].shape[3 + e] - 1)
        eb, ee = cut(E[b], b, 1, E[b].shape[3 + b] - 1), cut(E[e], e, 1, E[e].shape[3 + e] - 1)
        inner += -k[b] * diff(ee, b) + k[e] * diff(eb, e)
    for d in range(3):
        for c in range(3):
            if c == d:
                continue
            low = cut(torch.roll(B[c], 1, d), d, patch[d], patch[d] + os_).clone()
            high = cut(torch.roll(B[c], -1, d), d, os_ + 2, 2 * os_ + 2).clone()
            cut(B[c], d, 0, os_).copy_(low)
            cut(B[c], d, patch[d] + os_ + 2, patch[d] + 2 * os_ + 2).copy_(high)
    u, w = s["u"], s["w"]
    gam = torch.sqrt(1 + u[0] ** 2 + u[1] ** 2 + u[2] ** 2)
    x = [torch.remainder(s["x"][d] + dt * u[d] / gam, n[d] * dx[d]) for d in range(3)]
    cell = [torch.clamp((x[d] / dx[d]).long(), max=n[d] - 1) for d in range(3)]
    p, cl, lc = 0, 0, 0
    for d in range(3):
        inner = cell[d] % patch[d]
        p = p * npatch[d] + cell[d] // patch[d]
        cl = cl * (patch[d] // 4) + inner // 4
        lc = lc * 4 + inner % 4
    order = torch.argsort(p * math.prod(patch) + cl * 64 + lc, stable=True)
    return {"J": flat(J), "E": flat(E), "B": flat(B), "x": [t[order] for t in x], "u": [t[order] for t in u],
            "w": w[order], "charge": None, "key": None, "count": None, "ends": None}


def exact(case, seed):
    if case["kind"] == "sim":
        n, _ = _cells_dx(case)
        cost = math.prod(n) * case["ppc"] * case["steps"] * (3.0 if case["order"] == 4 else 1.0)
        if case["plasma"] == "resident" or cost > 6e7:
            return None
        return _exact_sim(case, seed)
    return {"patch": _exact_patch, "seam": _exact_seam, "patches": _exact_patches}[case["kind"]](case, seed)
