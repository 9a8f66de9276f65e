"""Workloads of this package as its users run them, for timing.

Each case is a plain dict.  prepare(case, seed) builds what a program holds
before the call (device grids with their states, batches, hierarchies, host
arrays), run(state) makes one pass through the public entry points, work(case)
gives the bytes and flops a pass cannot do without and exact(case, seed) gives
the same outputs in FP64 torch, without the package's code.

The kinds:
  loop     the reference's host loop on a device grid: cfl_dt_3d, then
           euler3d_step_, each returning finished (Sod tubes, Sedov blasts);
  host     the same loop on a numpy array, as a program with host arrays has it;
  rhs      euler3d_rhs_ on numpy arrays (dU and the three flux arrays);
  box      Batch.run on one turbulent box: device dt, the step as a hipGraph;
  batch    Batch.run on uneven independent Sod tubes and Sedov blasts;
  fmr      FMRHierarchy.run on a polytrope star with a static potential, two or
           three levels;
  binary   the coupled step: gas forces on two bodies, point masses, sinks,
           self-gravity every stage, accretion.
Sizes are cells per axis.  prec is the grid's form: "fp64" or "split".
"""
import ctypes as C
import importlib.util
import math
import pathlib
import sys

import numpy as np
import torch

NG = 3
XOFF = 13          # padded cell 0 of a device row sits 13 doubles into it
FLOORS = (1e-8, 1e-8)
CFL = 0.4


def _package():
    name = "binary_supernova_amd"
    if name not in sys.modules:
        d = pathlib.Path(__file__).resolve().parents[1] / "binary-supernova_amd"
        spec = importlib.util.spec_from_file_location(name, d / "__init__.py",
                                                      submodule_search_locations=[str(d)])
        sys.modules[name] = mod = importlib.util.module_from_spec(spec)
        spec.loader.exec_module(mod)
    return sys.modules[name]


def listed():
    return [
        # the reference's smallest run: latency of two synchronous calls
        dict(name="tube_128x8x8_fp64", kind="loop", what="tube", prec="fp64", nx=128, ny=8, nz=8),
        # an odd, ragged grid in the same loop
        dict(name="blast_97x61x45_fp64", kind="loop", what="blast", prec="fp64", nx=97, ny=61, nz=45),
        # a program whose state is a host array: both copies count
        dict(name="host_64_fp64", kind="host", what="blast", prec="fp64", nx=64, ny=64, nz=64),
        # the right-hand side as the generic RK3 driver calls it
        dict(name="rhs_48x40x36_fp64", kind="rhs", what="box", prec="fp64", nx=48, ny=40, nz=36),
        # the benchmark box, the largest pass
        dict(name="box_256_split", kind="box", what="box", prec="split", nx=256, ny=256, nz=256, steps=2),
        # the same physics in plain FP64
        dict(name="box_192_fp64", kind="box", what="box", prec="fp64", nx=192, ny=192, nz=192, steps=1),
        # a mid-size box no tile divides
        dict(name="box_100x75x130_split", kind="box", what="box", prec="split", nx=100, ny=75, nz=130, steps=4),
        # 48 uneven problems in one launch per kernel
        dict(name="batch_48_split", kind="batch", prec="split", count=48, lo=32, hi=128, steps=2),
        # a smaller batch in FP64
        dict(name="batch_12_fp64", kind="batch", prec="fp64", count=12, lo=32, hi=96, steps=2),
        # three nested levels at the benchmark's sizes: 192^3, 96^3, 128x128x96
        dict(name="fmr3_192_split", kind="fmr", prec="split", base=192, levels=3, ratio=2, steps=1),
        # the reference's two-level grid at a test's size: launches count
        dict(name="fmr2_32_fp64", kind="fmr", prec="fp64", base=32, levels=2, ratio=2, steps=1),
        # the binary run's coupled step on its fiducial 128^3
        dict(name="binary_128_split", kind="binary", prec="split", nx=128, ny=128, nz=128),
    ]


def _log(rng, lo, hi):
    return int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))


def draw(rng):
    kind = rng.choice(["loop", "loop", "host", "rhs", "box", "box", "batch", "fmr", "binary"])
    prec = rng.choice(["fp64", "split"])
    n = lambda lo, hi: dict(zip(("nx", "ny", "nz"), (_log(rng, lo, hi) for _ in range(3))))
    if kind == "loop":
        return dict(kind=kind, what=rng.choice(["tube", "blast"]), prec=prec, **n(6, 160))
    if kind == "host":
        return dict(kind=kind, what=rng.choice(["tube", "blast"]), prec="fp64", **n(8, 96))
    if kind == "rhs":
        return dict(kind=kind, what=rng.choice(["box", "blast"]), prec="fp64", **n(8, 64))
    if kind == "box":
        return dict(kind=kind, what="box", prec=prec, **n(24, 190), steps=rng.randint(1, 2))
    if kind == "batch":
        return dict(kind=kind, prec=prec, count=rng.randint(3, 24), lo=16, hi=rng.randint(48, 112), steps=rng.randint(1, 2))
    if kind == "fmr":
        # boxes of a third of the parent need a base of at least 24 cells
        return dict(kind=kind, prec=prec, base=4 * _log(rng, 6, 24), levels=2, ratio=rng.choice([2, 4]), steps=1)
    return dict(kind=kind, prec=prec, **n(24, 120))


# ---------------------------------------------------------------------------
# Inputs.  States are built on the GPU in the reference layout (Nz, Ny, Nx, 5).

def _gen(seed):
    return torch.Generator(device="cuda").manual_seed(int(seed))


def _field(n, gen, kmin=2.0, kmax=32.0):
    """Gaussian random field of P(k) ~ k^-11/3, zero mean, unit variance."""
    nz, ny, nx = n
    f = lambda m: torch.fft.fftfreq(m, d=1.0 / m, dtype=torch.float64, device="cuda")
    kx = torch.fft.rfftfreq(nx, d=1.0 / nx, dtype=torch.float64, device="cuda")
    kk = (f(nz)[:, None, None] ** 2 + f(ny)[None, :, None] ** 2 + kx[None, None, :] ** 2).sqrt()
    amp = torch.where((kk >= kmin) & (kk <= kmax), kk.clamp(min=1.0) ** (-11.0 / 6.0), torch.zeros_like(kk))
    w = torch.randn((2,) + tuple(kk.shape), generator=gen, dtype=torch.float64, device="cuda")
    s = torch.fft.irfftn(torch.complex(w[0] * amp, w[1] * amp), s=(nz, ny, nx))
    s = s - s.mean()
    return s / s.std()


def _conserved(rho, v, p, g):
    """(5, nz, ny, nx) conserved state from primitives."""
    return torch.stack([rho, rho * v[0], rho * v[1], rho * v[2],
                        p / (g - 1) + 0.5 * rho * (v[0] ** 2 + v[1] ** 2 + v[2] ** 2)])


def _axes(n, d, o):
    x, y, z = (o[a] + (torch.arange(n[a], dtype=torch.float64, device="cuda") + 0.5) * d[a] for a in range(3))
    return x[None, None, :], y[None, :, None], z[:, None, None]


def _problem(what, n, seed):
    """(active state, cell sizes, gamma, bc) of one problem on the unit cube."""
    r = np.random.default_rng(int(seed) & 0xffffffff)
    gen = _gen(seed)
    nx, ny, nz = n
    shape, d = (nz, ny, nx), (1.0 / nx, 1.0 / ny, 1.0 / nz)
    one, zero = torch.ones(shape, dtype=torch.float64, device="cuda"), torch.zeros((3,) + shape, dtype=torch.float64, device="cuda")
    if what == "box":       # supersonic turbulence, rms Mach 2, periodic
        g = 5.0 / 3.0
        rho = torch.exp(0.5 * _field(shape, gen))
        v = [_field(shape, gen) for _ in range(3)]
        m2 = (v[0] ** 2 + v[1] ** 2 + v[2] ** 2) * rho / g
        k = 2.0 / float(m2.mean().sqrt())
        return _conserved(rho, [k * a for a in v], one, g), d, g, "periodic"
    g = float(r.choice([1.4, 5.0 / 3.0]))
    if what == "tube":      # left and right states log-uniform on [0.1, 10]
        a = int(np.argmax(n))
        rl, rr, pl, pr = (float(q) for q in 10.0 ** r.uniform(-1, 1, 4))
        left = (_axes(n, d, (-0.5,) * 3)[a] < 0) & (one > 0)
        return _conserved(torch.where(left, rl, rr), zero, torch.where(left, pl, pr), g), d, g, "outflow"
    # a blast of log-uniform energy within 2.5 cells of a point near the centre
    c = r.uniform(-0.1, 0.1, 3)
    x, y, z = _axes(n, d, (-0.5,) * 3)
    inside = ((x - c[0]) ** 2 + (y - c[1]) ** 2 + (z - c[2]) ** 2).sqrt() <= 2.5 * max(d)
    e0 = float(10.0 ** r.uniform(-1, 1)) / (float(inside.sum()) * d[0] * d[1] * d[2])
    p = torch.where(inside, 1e-5 + e0 * (g - 1), 1e-5)
    return _conserved(one, zero, p, g), d, g, "outflow"


def _padded(A):
    """Reference layout (Nz, Ny, Nx, 5) with zero ghosts."""
    U = torch.zeros(tuple(m + 2 * NG for m in A.shape[1:]) + (5,), dtype=torch.float64, device="cuda")
    U[NG:-NG, NG:-NG, NG:-NG] = A.permute(1, 2, 3, 0)
    return U


def _load(g, A):
    """The device grid g takes the active state A from a device array."""
    U = _padded(A)
    torch.cuda.synchronize()
    _package()._lib.call("bsn_grid_set_state", g.handle, C.c_void_p(U.data_ptr()), 1)


class _Raw:
    """A grid's state buffer for torch; the tensor keeps this object, and it
    the grid, whose memory would otherwise go with the caller's last name for it."""

    def __init__(self, grid, ptr, n):
        self.grid = grid
        self.__cuda_array_interface__ = dict(shape=(n,), typestr="<f8", data=(ptr, False), version=2)


def _view(g):
    """The grid's own device state, active cells, (5, nz, ny, nx)."""
    p, fs, pitch = C.c_void_p(), C.c_int64(), C.c_int64()
    _package()._lib.call("bsn_grid_device_state", g.handle, C.byref(p), C.byref(fs), C.byref(pitch))
    raw = torch.as_tensor(_Raw(g, p.value, 5 * fs.value), device="cuda")
    Ny = g.ny + 2 * NG
    return torch.as_strided(raw, (5, g.nz, g.ny, g.nx), (fs.value, Ny * pitch.value, pitch.value, 1),
                            (NG * Ny + NG) * pitch.value + XOFF + NG)


def _dims(case):
    return case["nx"], case["ny"], case["nz"]


def _batch_sizes(case):
    """Sizes of the batch's problems: part of the case, not of the seed."""
    r = np.random.default_rng(case["count"] * 1000 + case["hi"])
    return [tuple(int(v) for v in r.integers(case["lo"], case["hi"] + 1, 3)) for _ in range(case["count"])]


def _batch_problems(case, seed):
    return [_problem(("tube", "blast")[k % 2], n, 1000 * (seed + 1) + k) for k, n in enumerate(_batch_sizes(case))]


def _fmr_geometry(case):
    """(dims, cell sizes, left edges, boxes): every child covers the middle
    third to half of its parent."""
    b, r, half = case["base"], case["ratio"], 8.0
    if case["levels"] == 3:
        # the benchmark star: 96^3 over a quarter, then 128 x 128 x 96 of it
        dims = [(b,) * 3, (b // 2,) * 3, (2 * b // 3, 2 * b // 3, b // 2)]
    else:
        # a third of the base per axis, an odd part longer in z
        w = max(6, b // 3 // 2 * 2)
        dims = [(b,) * 3, (r * w, r * w, r * (w + 2))]
    dx = [2 * half / b / r ** l for l in range(len(dims))]
    if case["levels"] == 2:
        dx = [0.25 * v for v in dx]
        half = 0.25 * half
    edges, boxes = [(-half,) * 3], []
    for l in range(1, len(dims)):
        lo = [(dims[l - 1][a] - dims[l][a] // r) // 2 + 1 for a in range(3)]
        boxes.append(tuple(v for a in range(3) for v in (lo[a], lo[a] + dims[l][a] // r - 1)))
        edges.append(tuple(edges[-1][a] + (lo[a] - 1) * dx[l - 1] for a in range(3)))
    return dims, [(v,) * 3 for v in dx], edges, boxes


def _star(n, d, o, gamma, seed, floor=(1e-10, 1e-12)):
    """Polytrope of unit radius and central density at the origin, with a few
    per cent of seeded large-scale noise in its density."""
    P = _package().problems
    xis, ths, _ = P.lane_emden(1.0 / (gamma - 1.0))
    _, r_scale, K, xi1 = P.polytrope_scales(gamma, 1.0, 1.0)
    x, y, z = _axes(n, d, o)
    q = (x * x + y * y + z * z).sqrt() / r_scale
    t = torch.tensor(ths, dtype=torch.float64, device="cuda")
    u = (q / (xis[1] - xis[0]) - 1.0).clamp(0, len(ths) - 1.001)
    i = u.floor().long()
    th = torch.where(q < xi1, (t[i] + (u - i) * (t[i + 1] - t[i])).clamp(min=0), 0.0)
    r = np.random.default_rng(int(seed) & 0xffffffff)
    k, ph = r.uniform(1, 4, 3), r.uniform(0, 6.28, 3)
    noise = 1 + 0.03 * torch.sin(k[0] * x + ph[0]) * torch.sin(k[1] * y + ph[1]) * torch.sin(k[2] * z + ph[2])
    nn = 1.0 / (gamma - 1.0)
    rho = torch.where(th > 0, (th ** nn * noise).clamp(min=floor[0]), floor[0])
    p = torch.where(th > 0, (K * rho ** (1 + 1 / nn)).clamp(min=floor[1]), floor[1])
    return _conserved(rho, torch.zeros((3,) + tuple(rho.shape), dtype=torch.float64, device="cuda"), p, gamma)


def _plummer(n, d, o):
    """Static potential of two point masses of 0.5 at (+-2, 0, 0), softening 0.1."""
    x, y, z = _axes(n, d, o)
    return sum(-0.5 / ((x - s) ** 2 + y * y + z * z + 0.01).sqrt() for s in (2.0, -2.0))


def _bodies(d):
    B = _package().BlackHole
    return [B(pos=[0.0, 0.0, 0.0], vel=[0.0, 0.0, 0.0], mass=0.5, eps=d[0], c_code=1e3, r_floor=2.5 * d[0]),
            B(pos=[1.2, 0.0, 0.0], vel=[0.0, 0.9, 0.0], mass=0.3, eps=d[0], c_code=1e3, r_floor=2.5 * d[0])]


STAR_FLOORS = (1e-10, 1e-12)


def _binary_setup(case):
    n = _dims(case)
    d = tuple(4.0 / m for m in n)
    return n, d, (-2.0,) * 3, 2e-4


def prepare(case, seed):
    bsn = _package()
    kind = case["kind"]
    if kind in ("loop", "host", "rhs"):
        n = _dims(case)
        A, d, g, bc = _problem(case["what"], n, seed)
        s = dict(kind=kind, n=n, d=d, g=g, bc=bc)
        if kind == "loop":
            s["grid"] = bsn.Grid(*n, case["prec"])
            _load(s["grid"], A)
            s["out"] = _view(s["grid"])
        else:
            s["U"] = _padded(A).cpu().numpy()
            if kind == "rhs":
                fx, fy, fz = bsn.flux_shapes(*n)
                s["outs"] = [np.zeros(s["U"].shape), np.zeros(fx), np.zeros(fy), np.zeros(fz)]
        return s
    if kind in ("box", "batch"):
        probs = [_problem("box", _dims(case), seed)] if kind == "box" else _batch_problems(case, seed)
        grids = []
        for A, d, g, bc in probs:
            grids.append(bsn.Grid(*A.shape[:0:-1], case["prec"]))
            _load(grids[-1], A)
            grids[-1].set_params(*d, g, bc, *FLOORS)
        return dict(kind="run", what=bsn.Batch(grids), steps=case["steps"], out=[_view(g) for g in grids])
    if kind == "fmr":
        dims, ds, edges, boxes = _fmr_geometry(case)
        g = 4.0 / 3.0
        H = bsn.FMRHierarchy(dims, ds, boxes, [case["ratio"]] * len(boxes), g, "outflow", *STAR_FLOORS, precision=case["prec"])
        for l, (n, d, o) in enumerate(zip(dims, ds, edges)):
            _load(H.levels[l], _star(n, d, o, g, seed))
            phi = _plummer(n, d, o).contiguous()
            torch.cuda.synchronize()
            bsn._lib.call("bsn_grid_set_phi", H.levels[l].handle, C.c_void_p(phi.data_ptr()), 1)
        return dict(kind="run", what=H, steps=case["steps"], out=[_view(g) for g in H.levels])
    n, d, o, dt = _binary_setup(case)
    grid = bsn.Grid(*n, case["prec"])
    _load(grid, _star(n, d, o, 5.0 / 3.0, seed))
    grid.set_params(*d, 5.0 / 3.0, "outflow", *STAR_FLOORS)
    b = bsn.Batch([grid])
    bsn.set_self_gravity(grid, True)
    return dict(kind=kind, n=n, d=d, o=o, dt=dt, grid=grid, batch=b, bhs=_bodies(d), out=_view(grid))


def run(s):
    bsn = _package()
    kind = s["kind"]
    if kind == "run":
        s["what"].run(CFL, s["steps"], graph=True)
        return s["out"]
    n, d = s["n"], s["d"]
    if kind == "binary":
        grid, bhs, o = s["grid"], s["bhs"], s["o"]
        F = bsn.gas_forces_on_bhs(grid, *n, *d, bhs, *o)
        for bh, f in zip(bhs, F):
            for c in range(3):
                bh.vel[c] += s["dt"] * f[c] / bh.mass
                bh.pos[c] += s["dt"] * bh.vel[c]
        bsn.set_point_masses(grid, bhs, *o)
        bsn.set_sinks(grid, bhs, *o, f_sink=1.0, torque_free=True, rho_sink_min=1e-6)
        s["batch"].step([s["dt"]])
        dm = bsn.accrete_all_(bhs, grid, *n, *d, *o, s["dt"], rho_sink_min=1e-6)
        return [s["out"], F, dm]
    g, bc = s["g"], s["bc"]
    if kind == "rhs":
        bsn.euler3d_rhs_(*s["outs"], s["U"], *n, *d, g, bc=bc, rho_floor=FLOORS[0], P_floor=FLOORS[1])
        return s["outs"]
    U = s["grid"] if kind == "loop" else s["U"]
    dt = bsn.cfl_dt_3d(U, *n, *d, g, CFL)
    bsn.euler3d_step_(U, *n, *d, dt, g, bc=bc, rho_floor=FLOORS[0], P_floor=FLOORS[1])
    return [s["out"] if kind == "loop" else s["U"][NG:-NG, NG:-NG, NG:-NG], dt]


# Per cell and RK3 step: the FP64 state read and written each stage and the
# base state in two of them (320 B); three interfaces a stage at 784 flops each
# (a division or square root as one).
STEP_BYTES, STEP_FLOPS = 320, 3 * 3 * 784


def work(case):
    kind = case["kind"]
    if kind == "batch":
        cells = sum(a * b * c for a, b, c in _batch_sizes(case)) * case["steps"]
    elif kind == "fmr":
        dims = _fmr_geometry(case)[0]
        cells = sum(a * b * c * case["ratio"] ** l for l, (a, b, c) in enumerate(dims)) * case["steps"]
    else:
        cells = case["nx"] * case["ny"] * case["nz"] * case.get("steps", 1)
    if kind == "rhs":       # the state in, dU and three flux arrays out
        return dict(bytes=200 * cells, flops=3 * 784 * cells)
    if kind == "binary":
        # per stage a real transform of the 8 times larger padded density and
        # back, the density read and phi written and read again
        big = 8 * cells
        return dict(bytes=(STEP_BYTES + 3 * 24) * cells, flops=STEP_FLOPS * cells + 3 * 2 * 2.5 * big * math.log2(big))
    return dict(bytes=(STEP_BYTES + (24 if kind == "fmr" else 0)) * cells, flops=STEP_FLOPS * cells)


# ---------------------------------------------------------------------------
# The same in plain FP64 torch: active states (5, nz, ny, nx), axis a = x, y, z.

def _weno(a):
    """Left and right WENO5-Z values at the interface between a[2] and a[3]."""
    A = lambda x, y, z: 13 / 12 * (x - 2 * y + z) ** 2 + 0.25 * (x - 4 * y + 3 * z) ** 2
    B = lambda x, y, z: 13 / 12 * (x - 2 * y + z) ** 2 + 0.25 * (x - z) ** 2
    D = lambda x, y, z: 13 / 12 * (x - 2 * y + z) ** 2 + 0.25 * (3 * x - 4 * y + z) ** 2

    def mix(b, w, q):
        tau = (b[0] - b[2]).abs()
        al = [wi * (1 + (tau / (1e-36 + bi)) ** 2) for wi, bi in zip(w, b)]
        s = al[0] + al[1] + al[2]
        return sum(x / s * y for x, y in zip(al, q))
    q0 = a[0] / 3 - 7 / 6 * a[1] + 11 / 6 * a[2]
    qc = -a[1] / 6 + 5 / 6 * a[2] + a[3] / 3
    qr = a[2] / 3 + 5 / 6 * a[3] - a[4] / 6
    q2 = 11 / 6 * a[3] - 7 / 6 * a[4] + a[5] / 3
    L = mix((A(*a[:3]), B(*a[1:4]), D(*a[2:5])), (0.1, 0.6, 0.3), (q0, qc, qr))
    # the right side's middle indicator is one-sided, as the reference has it
    return L, mix((B(*a[1:4]), A(*a[2:5]), D(*a[3:])), (0.3, 0.6, 0.1), (qc, qr, q2))


def _hllc(L, R, n, g):
    """HLLC flux of (rho, m, P) states along momentum n, P turned into E."""
    def energy(u):
        r = u[0].clamp(min=1e-30)
        ke = torch.minimum(0.5 * (u[1] ** 2 + u[2] ** 2 + u[3] ** 2) / r, 0.5e4 * r)
        return u[4] / (g - 1) + ke

    def side(u):
        E = energy(u)
        ok = u[0] > 0
        r = torch.where(ok, u[0].clamp(min=1e-30), 1e-30)
        m = [torch.where(ok, x, 0.0) for x in u[1:4]]
        E = torch.where(ok, E, 0.0)
        m2 = m[0] ** 2 + m[1] ** 2 + m[2] ** 2
        k = torch.where(m2 > 1e4 * r * r, 100 * r / m2.clamp(min=1e-300).sqrt(), 1.0)
        m = [k * x for x in m]
        ke = torch.minimum(0.5 * (m[0] ** 2 + m[1] ** 2 + m[2] ** 2) / r, 0.5e4 * r)
        E = torch.maximum(E, ke)
        p = (g - 1) * (E - ke)
        v = m[n] / r
        F = [m[n]] + [x * v for x in m] + [(E + p) * v]
        F[1 + n] = r * v * v + p
        return r, m, E, p, v, (g * p / r).sqrt(), F
    rL, mL, EL, pL, vL, cL, FL = side(L)
    rR, mR, ER, pR, vR, cR, FR = side(R)
    ps = (0.5 * (pL + pR) - 0.5 * (vR - vL) * 0.5 * (rL + rR) * 0.5 * (cL + cR)).clamp(min=0)
    fac = (g + 1) / (2 * g)
    q = lambda p: torch.where(ps > p, (1 + fac * (ps / p - 1).clamp(min=0)).sqrt(), 1.0)
    pos = (pL > 0) & (pR > 0)
    SL = torch.where(pos, vL - cL * q(pL), torch.minimum(vL - cL, vR - cR))
    SR = torch.where(pos, vR + cR * q(pR), torch.maximum(vL + cL, vR + cR))
    den = rL * (SL - vL) - rR * (SR - vR)
    S = (pR - pL + rL * vL * (SL - vL) - rR * vR * (SR - vR)) / den
    hll = torch.maximum(rL, rR) > 3 * torch.minimum(rL, rR)
    left = S >= 0
    r, E, p, v, K = (torch.where(left, x, y) for x, y in ((rL, rR), (EL, ER), (pL, pR), (vL, vR), (SL, SR)))
    m = [torch.where(left, x, y) for x, y in zip(mL, mR)]
    dk = r * (K - v)
    chi = dk / (K - S)
    star = [chi] + [chi * x / r for x in m] + [torch.where(dk.abs() > 1e-100, chi * (E / r + (S - v) * (S + p / dk)), 0.0)]
    star[1 + n] = chi * S
    uL, uR = [rL] + mL + [EL], [rR] + mR + [ER]
    out = []
    for c in range(5):
        h = (SR * FL[c] - SL * FR[c] + SL * SR * (uR[c] - uL[c])) / (SR - SL)
        k = torch.where(left, FL[c], FR[c]) + K * (star[c] - torch.where(left, uL[c], uR[c]))
        f = torch.where(hll, h, k)
        f = torch.where(SR <= 0, FR[c], f)
        f = torch.where(SL >= 0, FL[c], f)
        out.append(torch.where(den.abs() < 1e-100, 0.0, f))
    return torch.stack(out)


def _pressure(U, g):
    return ((g - 1) * (U[4] - 0.5 * (U[1] ** 2 + U[2] ** 2 + U[3] ** 2) / U[0].clamp(min=1e-30))).clamp(min=0)


def _fluxes(P, g):
    """Interface fluxes of the padded state P along x, y and z."""
    out = []
    for a in range(3):
        dim = 3 - a
        Q = P
        for o in (1, 2, 3):
            if o != dim:
                Q = Q.narrow(o, NG, Q.shape[o] - 2 * NG)
        W = [Q[c] for c in range(4)] + [_pressure(Q, g)]
        L, R = [], []
        for c, w in enumerate(W):
            s = [w.narrow(dim - 1, k, w.shape[dim - 1] - 5) for k in range(6)]
            l, r = _weno(s)
            if c == 4:
                top = lambda t: torch.stack(t).amax(0)
                l, r = torch.minimum(l.clamp(min=0), top(s[:5])), torch.minimum(r.clamp(min=0), top(s[1:]))
            L.append(l)
            R.append(r)
        out.append(_hllc(L, R, a, g))
    return out


def _floor(U, g, rf, pf):
    low = U[0] < rf
    ke = 0.5 * (U[1] ** 2 + U[2] ** 2 + U[3] ** 2) / U[0]
    E = torch.where((g - 1) * (U[4] - ke) < pf, pf / (g - 1) + ke, U[4])
    V = torch.cat([U[:4], E[None]])
    V = torch.where(low, 0.0, V)
    V[0] = torch.where(low, rf, V[0])
    V[4] = torch.where(low, pf / (g - 1), V[4])
    return V


def _pad(U, bc):
    for dim in (3, 2, 1):
        n = U.shape[dim]
        i = torch.arange(-NG, n + NG, device=U.device)
        U = U.index_select(dim, i % n if bc == "periodic" else i.clamp(0, n - 1))
    return U


def _speed(U, d, g):
    r = U[0].clamp(min=1e-30)
    c = (g * _pressure(U, g) / r).sqrt()
    return max(float(((U[1 + a] / r).abs() + c).max()) / d[a] for a in range(3))


def _divergence(F, d):
    D = 0.0
    for a in range(3):
        n = F[a].shape[3 - a] - 1
        D = D - (F[a].narrow(3 - a, 1, n) - F[a].narrow(3 - a, 0, n)) / d[a]
    return D


def _add_phi(D, U, phi, d):
    dot = 0.0
    for a in range(3):
        dim = 2 - a
        n = phi.shape[dim]
        i = torch.arange(n, device=phi.device)
        gr = (phi.index_select(dim, (i + 1).clamp(max=n - 1)) - phi.index_select(dim, (i - 1).clamp(min=0))) * (0.5 / d[a])
        D[1 + a] -= U[0] * gr
        dot = dot + U[1 + a] * gr
    D[4] -= dot
    return D


def _combine(s, Un, U, D, dt):
    w = ((1.0, 0.0, 1.0), (0.75, 0.25, 0.25), (1 / 3, 2 / 3, 2 / 3))[s]
    return w[0] * Un + w[1] * U + w[2] * dt * D


def _step(U, d, dt, g, bc, floors, source=None):
    """One SSP-RK3 step; source(D, U) adds to each stage's right-hand side."""
    Un = U
    for s in range(3):
        P = _pad(U, bc)
        if s == 0:
            U = _floor(U, g, *floors)
            P = P.clone()
            P[:, NG:-NG, NG:-NG, NG:-NG] = U
        D = _divergence(_fluxes(P, g), d)
        if source is not None:
            D = source(D, U)
        U = _floor(_combine(s, Un, U, D, dt), g, *floors)
    return U


def _poisson(rho, d):
    n = rho.shape[::-1]
    r2 = 0.0
    for a in range(3):
        i = torch.arange(2 * n[a], dtype=torch.float64, device="cuda")
        i = torch.where(i < n[a], i, i - 2 * n[a]) * d[a]
        r2 = r2 + (i ** 2).reshape([-1 if 2 - a == k else 1 for k in range(3)])
    dV = d[0] * d[1] * d[2]
    big = tuple(2 * m for m in rho.shape)
    K = torch.fft.rfftn(-1 / (r2 + dV ** (2 / 3)).sqrt())
    phi = torch.fft.irfftn(K * torch.fft.rfftn(rho, s=big), s=big) * dV
    return phi[:rho.shape[0], :rho.shape[1], :rho.shape[2]].contiguous()


def _exact_binary(case, seed):
    n, d, o, dt = _binary_setup(case)
    g = 5.0 / 3.0
    U = _star(n, d, o, g, seed)
    x, y, z = X = _axes(n, d, o)
    dV = d[0] * d[1] * d[2]
    b = _bodies(d)
    sep = lambda p: [X[c] - p[c] for c in range(3)]
    F = []
    for h in b:
        e = sep(h.pos)
        w = U[0] * h.mass / (e[0] ** 2 + e[1] ** 2 + e[2] ** 2 + h.eps ** 2) ** 1.5
        F.append([float((w * q).sum()) * dV for q in e])
    for h, f in zip(b, F):
        for c in range(3):
            h.vel[c] += dt * f[c] / h.mass
            h.pos[c] += dt * h.vel[c]
    rs = [max(6 * h.mass / h.c_code ** 2, h.r_floor) for h in b]
    ts = [r / math.sqrt(2 * h.mass / r) for r, h in zip(rs, b)]

    def source(D, U):
        v = [U[1 + c] / U[0] for c in range(3)]
        for h in b:
            e = sep(h.pos)
            k = -h.mass / (e[0] ** 2 + e[1] ** 2 + e[2] ** 2 + h.eps ** 2) ** 1.5
            for c in range(3):
                D[1 + c] += U[0] * k * e[c]
                D[4] += U[1 + c] * k * e[c]
        D = _add_phi(D, U, _poisson(U[0], d), d)
        for h, r, t in zip(b, rs, ts):
            e = sep(h.pos)
            dist = (e[0] ** 2 + e[1] ** 2 + e[2] ** 2).sqrt()
            on = ((dist < r) & (U[0] > 1e-6)).double() / t
            u = [q / dist.clamp(min=1e-300) for q in e]
            vr = sum((v[c] - h.vel[c]) * u[c] for c in range(3))
            D[0] -= on * U[0]
            for c in range(3):
                D[1 + c] -= on * U[0] * vr * u[c]
            eint = U[4] / U[0] - 0.5 * (v[0] ** 2 + v[1] ** 2 + v[2] ** 2)
            D[4] -= on * (0.5 * U[0] * vr ** 2 + U[0] * eint)
        return D
    U = _step(U, d, dt, g, "outflow", STAR_FLOORS, source)
    dm = []
    for h, r, t in zip(b, rs, ts):
        e = sep(h.pos)
        on = ((e[0] ** 2 + e[1] ** 2 + e[2] ** 2).sqrt() < r) & (U[0] > 1e-6)
        dm.append(float(torch.where(on, U[0], 0.0).sum()) * dV / t * dt)
    return [U, np.array(F), np.array(dm)]


def _prolong(P, lo, ratio, nf):
    """Every padded fine cell from the padded parent P: 5-point Lagrange per axis."""
    for a in (2, 1, 0):
        dim = 3 - a
        i = torch.arange(1, nf[a] + 2 * NG + 1, dtype=torch.float64)
        xi = lo[a] - 0.5 + (i - NG - 0.5) / ratio
        c = xi.round()
        s = ((xi - c + 0.5) * ratio).floor().clamp(0, ratio - 1)
        t = (s + 0.5 - ratio / 2) / ratio
        out = 0.0
        for j in range(5):
            w = torch.ones_like(t)
            for m in range(5):
                if m != j:
                    w = w * (t - (m - 2)) / (j - m)
            w = w.to(P.device).reshape([-1 if k == dim else 1 for k in range(4)])
            out = out + w * P.index_select(dim, (c.long() + NG - 1 + j - 2).to(P.device))
        P = out
    return P


def _exact_fmr(case, seed):
    dims, ds, edges, boxes = _fmr_geometry(case)
    g, r, N = 4.0 / 3.0, case["ratio"], len(dims)
    U = [_star(n, d, o, g, seed) for n, d, o in zip(dims, ds, edges)]
    phi = [_plummer(n, d, o) for n, d, o in zip(dims, ds, edges)]
    coarse, fine = [None] * N, [None] * N       # flux registers of level l's child
    core = (slice(None),) + (slice(NG, -NG),) * 3

    def box(l):
        b = boxes[l]
        return [slice(b[2 * a] - 1, b[2 * a + 1]) for a in range(3)]

    def advance(l, dt, ghosts):
        d, Un = ds[l], U[l]
        V = Un
        if l + 1 < N:
            coarse[l], fine[l] = [0.0] * 6, [0.0] * 6
        for s, w in enumerate((1 / 6, 1 / 6, 2 / 3)):
            P = _pad(V, "outflow") if l == 0 else ghosts.clone()
            if s == 0:
                V = _floor(V, g, *STAR_FLOORS)
            P = P.clone()
            P[core] = V
            F = _fluxes(P, g)
            if l + 1 < N:
                bx = box(l)
                for a in range(3):
                    for e, f in enumerate((bx[a].start, bx[a].stop)):
                        t = F[a].narrow(3 - a, f, 1)
                        for k in range(3):
                            if k != a:
                                t = t.narrow(3 - k, bx[k].start, bx[k].stop - bx[k].start)
                        coarse[l][2 * a + e] = coarse[l][2 * a + e] + w * dt * t
            if l > 0:
                for a in range(3):
                    for e, f in enumerate((0, dims[l][a])):
                        t = F[a].narrow(3 - a, f, 1)
                        for k in range(3):
                            if k != a:
                                t = t.unflatten(3 - k, (-1, r)).sum(4 - k)
                        fine[l - 1][2 * a + e] = fine[l - 1][2 * a + e] + w * dt / r ** 2 * t
            D = _add_phi(_divergence(F, d), V, phi[l], d)
            V = _floor(_combine(s, Un, V, D, dt), g, *STAR_FLOORS)
        U[l] = V
        if l + 1 < N:
            b = boxes[l]
            for q in range(r):
                mix = (1 - q / r) * Un + q / r * V
                advance(l + 1, dt / r, _prolong(_pad(mix, "outflow"), b[::2], r, dims[l + 1]))
            V = V.clone()
            bx = box(l)
            child = U[l + 1]
            V[:, bx[2], bx[1], bx[0]] = child.unflatten(3, (-1, r)).unflatten(2, (-1, r)).unflatten(1, (-1, r)).mean((2, 4, 6))
            for a in range(3):
                for e, cell in enumerate((bx[a].start - 1, bx[a].stop)):
                    at = [slice(None)] + [bx[2], bx[1], bx[0]]
                    at[3 - a] = slice(cell, cell + 1)
                    jump = fine[l][2 * a + e] - coarse[l][2 * a + e]
                    V[tuple(at)] += (jump if e else -jump) / d[a]
            U[l] = _floor(V, g, *STAR_FLOORS)
    for _ in range(case["steps"]):
        dt = min(r ** l * CFL / _speed(U[l], ds[l], g) for l in range(N))
        advance(0, dt, None)
    return U


def exact(case, seed):
    kind = case["kind"]
    if kind == "fmr":
        return _exact_fmr(case, seed)
    if kind == "binary":
        return _exact_binary(case, seed)
    if kind == "batch":
        probs = _batch_problems(case, seed)
    else:
        probs = [_problem(case["what"], _dims(case), seed)]
    out = []
    for U, d, g, bc in probs:
        if kind == "rhs":
            V = _floor(U, g, *FLOORS)
            P = _pad(U, bc).clone()
            P[:, NG:-NG, NG:-NG, NG:-NG] = V
            F = _fluxes(P, g)
            return [_reference(_divergence(F, d), V.shape, None)] + [_reference(F[a], V.shape, a) for a in range(3)]
        for _ in range(case.get("steps", 1)):
            dt = CFL / _speed(U, d, g)
            U = _step(U, d, dt, g, bc, FLOORS)
        out.append(U)
    if kind == "loop":
        return [out[0], dt]
    if kind == "host":
        return [out[0].permute(1, 2, 3, 0).cpu().numpy(), dt]
    return out


def _reference(F, shape, a):
    """An active array or flux in the reference's padded layout, zero outside."""
    full = [m + 2 * NG for m in shape[1:]]
    at = [slice(NG, NG + m) for m in shape[1:]]
    if a is not None:       # interface f sits at 0-based index NG - 1 + f along its axis
        full[2 - a] += 1
        at[2 - a] = slice(NG - 1, NG + shape[3 - a])
    out = torch.zeros(tuple(full) + (5,), dtype=torch.float64, device="cuda")
    out[tuple(at)] = F.permute(1, 2, 3, 0)
    return out.cpu().numpy()
