"""The performance cases of the time-stepping core.

What a program that uses this framework has it do, each as one pass through
the public entry points of ``cgfd.model``:

* advance one rupture simulation between two outputs (``Core.run`` and the
  reads of that output), from the smallest grid to the largest, one step at a
  time or several;
* advance an ensemble of rupture scenarios on one grid (``Batch``);
* one gradient evaluation: restart, forward run with the friction tape, and
  the adjoint (``Core.adjoint_initial`` / ``adjoint_fault``, and a batch's).

Axes are the reference's: ni fault-normal, nj strike, nk depth. Sizes are
those of cgfd.configs, of the tests and of bench.py, and generic odd ones.
Grids, media and wavefields are made on the GPU from the seed; the initial
wavefield (waves all over the domain) enters as a checkpoint in device memory
(``load_state``), so a pass works on a developed wavefield.

``exact`` holds the waves alone (metric, stencil, CFS-PML, free surface, RK4,
and their adjoint by automatic differentiation) in 64 bits; it has no value
for the cases with a fault.
"""
from __future__ import annotations

import ctypes as C
import math
import sys
from pathlib import Path

import numpy as np
import torch

sys.path.insert(0, str(Path(__file__).resolve().parent.parent / "gpu-cgfd3d-dynamic_amd"))

from cgfd import lib as L  # noqa: E402
from cgfd import model  # noqa: E402

MPA = 1.0e6
DH = 100.0
DEV = "cuda"


def _case(name, kind, ni, nj, nk, pml, steps, grid="topo", method=2, faults=1, buried=False, out="state", nscen=1):
    c = {"kind": kind, "ni": ni, "nj": nj, "nk": nk, "pml": pml, "steps": steps, "grid": grid, "method": method,
         "faults": faults, "buried": buried, "out": out, "nscen": nscen}
    if name:
        c["name"] = name
    return c


def listed():
    return [
        # the smallest grid of the tests, a driver that writes slices, fault
        # frames and PG after every step: latency, launches, small reads
        _case("step_small", "forward", 36, 48, 28, 5, 1, out="frames"),
        # the CPU-runnable 120 x 80 x 60 half-space, ten steps between outputs
        # (one graph block of eight and two single steps)
        _case("flat_80x120x60", "forward", 80, 120, 60, 12, 10, grid="flat"),
        # odd sizes, two buried rough faults, method 1, six CFS-PML faces; no
        # metric term vanishes
        _case("rough_101x173x83", "forward", 101, 173, 83, 11, 7, grid="rough", method=1, faults=2, buried=True),
        # waves without a fault under topography on general curvilinear
        # columns (a velocity model's response to an initial field)
        _case("waves_96x141x72", "forward", 96, 141, 72, 10, 8, grid="rough", faults=0),
        # the differentiation grid, run forward
        _case("topo_160x240x100", "forward", 160, 240, 100, 12, 8),
        # one scenario of the ensemble grid
        _case("topo_200x400x150", "forward", 200, 400, 150, 20, 8),
        # the 1200 x 600 x 400 production run at two thirds of its linear
        # size: the largest
        _case("topo_400x800x266", "forward", 400, 800, 266, 20, 8),
        # a small ensemble
        _case("batch6_80x120x60", "batch", 80, 120, 60, 12, 8, nscen=6),
        # the ensemble grid with twelve of its scenarios
        _case("batch12_200x400x150", "batch", 200, 400, 150, 20, 4, nscen=12),
        # gradient of a trace misfit with respect to the initial field, no
        # fault: small, latency and launches count
        _case("grad_waves_50x71x40", "adjoint", 50, 71, 40, 6, 9, faults=0),
        # gradient through the rupture on the differentiation grid
        _case("grad_160x240x100", "adjoint", 160, 240, 100, 12, 17),
        # gradients of an ensemble's scenarios (the batched adjoint grid at
        # 0.4 of its linear size)
        _case("grad_batch3_80x128x48", "batch_adjoint", 80, 128, 48, 8, 9, nscen=3),
    ]


def _log_int(rng, lo, hi):
    return int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))


def draw(rng):
    kind = rng.choice(["forward"] * 5 + ["batch", "adjoint", "adjoint", "batch_adjoint"])
    most = {"forward": 60e6, "batch": 60e6, "adjoint": 4e6, "batch_adjoint": 1.5e6}[kind]
    nscen = rng.randint(2, 10) if kind.startswith("batch") else 1
    while True:
        ni, nj, nk = _log_int(rng, 36, 400), _log_int(rng, 46, 800), _log_int(rng, 28, 266)
        if ni * nj * nk * nscen <= most:
            break
    pml = min(20, max(5, min(ni // 6, nj // 7, nk // 5)))
    grid = rng.choice(["flat", "topo", "topo", "rough"])
    steps = rng.randint(1, 12) if not kind.endswith("adjoint") else rng.randint(4, 14)
    if ni * nj * nk * nscen > 2e7:
        steps = min(steps, 5)
    faults = 1 if kind.startswith("batch") else rng.choice([0, 1, 1, 1, 2])
    if faults == 2 and ni < 2 * pml + 34:
        faults = 1
    buried = rng.random() < 0.25
    out = rng.choice(["state", "state", "frames"]) if kind == "forward" else "state"
    return _case(None, kind, ni, nj, nk, pml, steps, grid, rng.choice([1, 2, 2]), faults, buried, out, nscen)


def work(case):
    """Bytes and operations a pass cannot do without. The grid does not stay
    on chip between the stages of a step, so per point and RK stage: the
    stage input once (36 B), the metric and media (8 arrays where the columns
    are vertical, 12 otherwise), the step's start and the earlier stages'
    outputs where the stage combines them, and one written level; 1.7 kFLOP
    per point and step. A reverse step reads and writes per stage as much as
    a forward stage (media, metric, two levels in, one out)."""
    per = 596 if case["grid"] != "rough" else 660
    n = case["ni"] * case["nj"] * case["nk"] * case["nscen"] * case["steps"]
    byts, flops = per * n, 1700 * n
    if case["kind"].endswith("adjoint"):
        byts += per * n
        flops += 1700 * n
    return {"bytes": byts, "flops": flops}


# ---------------------------------------------------------------------------
# inputs


def _axes(case, dtype=torch.float64):
    ni, nj, nk = case["ni"], case["nj"], case["nk"]
    i = torch.arange(ni, dtype=dtype, device=DEV)
    j = torch.arange(nj, dtype=dtype, device=DEV)
    k = torch.arange(nk, dtype=dtype, device=DEV)
    return i, j, k


def _x_index(case):
    """Fault planes' x indices."""
    mid = case["ni"] // 2
    return {0: [], 1: [mid], 2: [mid - 5, mid + 6]}[case["faults"]]


def _grid(case, rng):
    """(x, y, z, local topography) as float32 (nk, nj, ni) on the GPU: 100 m,
    hills up to 4 nodes high, the vertical spacing growing to 1.5 times at
    the bottom; "rough" also bends the constant-i planes (along strike and
    depth), so no metric term vanishes."""
    i, j, k = _axes(case)
    ni, nj, nk = case["ni"], case["nj"], case["nk"]
    x0, y0 = (i - ni // 2) * DH, (j - nj // 2) * DH
    topo = torch.zeros((nj, ni), dtype=torch.float64, device=DEV)
    if case["grid"] != "flat":
        for _ in range(4):
            h, w = rng.uniform(100.0, 400.0), rng.uniform(8.0, 40.0) * DH
            xc, yc = rng.uniform(-0.5, 0.5) * ni * DH, rng.uniform(-0.5, 0.5) * nj * DH
            topo += h * torch.exp(-((x0[None, :] - xc) ** 2 + (y0[:, None] - yc) ** 2) / (2.0 * w * w))
    if case["grid"] == "flat":
        zf = (k - (nk - 1)) * DH
    else:
        sp = DH * (1.0 + 0.5 * torch.arange(nk - 1, dtype=torch.float64, device=DEV) / max(nk - 2, 1))
        zf = torch.cat([torch.zeros(1, dtype=torch.float64, device=DEV), -torch.cumsum(sp, 0)]).flip(0)
    x = x0[None, None, :].expand(nk, nj, ni)
    y = y0[None, :, None].expand(nk, nj, ni)
    z = zf[:, None, None] + topo[None] * ((zf - zf[0]) / (0.0 - zf[0]))[:, None, None]
    if case["grid"] == "rough":
        a, b = rng.uniform(0.0, 6.28), rng.uniform(0.0, 6.28)
        bend = 0.8 * DH * (torch.sin(y0[None, :] / (17.0 * DH) + a) + torch.sin(zf[:, None] / (13.0 * DH) + b))
        x = x + bend[:, :, None]
        y = y + (0.5 * DH * torch.sin(zf / (15.0 * DH) + a))[:, None, None] + 0.0 * x0
    return x.float().contiguous(), y.float().contiguous(), z.float().contiguous(), topo


def _media(case, z, topo, seed):
    """Layered medium below the local surface with 3% noise."""
    g = torch.Generator(device=DEV).manual_seed(seed)
    depth = (topo[None].float() - z) / 1000.0
    vs = torch.full_like(z, 1.8)
    for t, v in ((1.0, 2.2), (3.0, 2.7), (6.0, 3.2), (10.0, 3.6)):
        vs[depth >= t] = v
    vp = 1.73 * vs
    rho = 1741.0 * vp ** 0.25
    f = 1.0 + 0.03 * torch.randn(z.shape, generator=g, device=DEV).clamp_(-3.0, 3.0)
    vs, vp, rho = 1000.0 * vs * f, 1000.0 * vp * f, rho * f
    mu = vs * vs * rho
    lam = vp * vp * rho - 2.0 * mu
    return lam, mu, rho


def _fault_fields(case, rng, plane):
    """Friction and initial stress of one fault and one scenario: strength
    0.68 sigma_n, 2% noise on the shear stress, a nucleation patch above its
    strength, the plane locked outside the fault's grid."""
    nj, nk, pml = case["nj"], case["nk"], case["pml"]
    f = {k: np.zeros((nk, nj), np.float32) for k in model.FAULT_FIELDS}
    j1, j2, k1, k2 = plane
    jj, kk = np.meshgrid(np.arange(nj), np.arange(nk))
    inside = (jj >= j1) & (jj <= j2) & (kk >= k1) & (kk <= k2)
    f["mu_s"][:] = np.where(inside, rng.uniform(0.66, 0.70, size=(nk, nj)), 1000.0)
    f["mu_d"][:] = 0.52
    f["Dc"][:] = rng.uniform(0.3, 0.5, size=(nk, nj))
    f["Tx"][:] = -120.0 * MPA
    f["Ty"][:] = 66.0 * MPA * (1.0 + rng.uniform(-0.02, 0.02, size=(nk, nj)))
    n = max(4, min(j2 - j1, k2 - k1) // 4)
    pj = int(rng.integers(j1 + 1, max(j2 - n, j1 + 2)))
    pk = int(rng.integers(k1 + 1, max(k2 - n, k1 + 2)))
    patch = inside & (jj >= pj) & (jj < pj + n) & (kk >= pk) & (kk < pk + n)
    f["Ty"][patch] = f["mu_s"][patch] * np.float32(120.0 * MPA) + np.float32(2.0 * MPA)
    return f


def _plane(case):
    nj, nk, pml = case["nj"], case["nk"], case["pml"]
    lo = pml + 4
    k2 = nk - 1 if not case["buried"] else nk - 1 - lo
    return lo, nj - 1 - lo, lo, k2


def _layers(case):
    p = case["pml"]
    return [[p, p], [p, p], [p, p if case["buried"] else 0]]


def _dt(case):
    return 0.006 if case["grid"] != "rough" else 0.005


def _scenario(case, seed):
    """(Scenario, fault fields per scenario)"""
    rng = np.random.default_rng(seed)
    x, y, z, topo = _grid(case, rng)
    lam, mu, rho = _media(case, z, topo, seed)
    planes = [_plane(case) for _ in _x_index(case)]
    fields = [[_fault_fields(case, rng, pl) for pl in planes] for _ in range(case["nscen"])]
    faults = [model.FaultSpec(x_index=i0, grid=pl, fields=f) for i0, pl, f in zip(_x_index(case), planes, fields[0])]
    h = [t.cpu().numpy() for t in (x, y, z, lam, mu, rho)]
    sc = model.Scenario(ni=case["ni"], nj=case["nj"], nk=case["nk"], x=h[0], y=h[1], z=h[2], lam=h[3], mu=h[4],
                        rho=h[5], free_top=not case["buried"], pml_layers=_layers(case), imethod=case["method"],
                        faults=faults, united_margin=case["pml"] + 3, dt=_dt(case), nt_total=10 ** 8)
    return sc, fields


def _stations(case, seed):
    """Receivers (ghost-inclusive nodes): 16, most of them on the surface."""
    rng = np.random.default_rng(seed + 77)
    n, p = 16, 3
    ijk = np.stack([rng.integers(p, case["ni"] - p, n), rng.integers(p, case["nj"] - p, n),
                    np.where(np.arange(n) % 4 == 3, case["nk"] // 2, case["nk"] - 1)], axis=1)
    return ijk.astype(np.int32) + 3


def _waves(case, seed, scale=1.0):
    """A wavefield (9, nz, ny, nx), ghosts zero, of four plane waves per
    component with wavelengths of 8 to 30 nodes, 2 cm/s and the stresses that
    go with it, fading towards the fault planes."""
    rng = np.random.default_rng(seed + 991)
    i, j, k = _axes(case, torch.float32)
    ni, nj, nk = case["ni"], case["nj"], case["nk"]
    w = torch.zeros((9, nk + 6, nj + 6, ni + 6), device=DEV)
    fade = torch.ones(ni, device=DEV)
    for i0 in _x_index(case):
        fade *= 1.0 - torch.exp(-((i - i0) / 6.0) ** 2)
    for c in range(9):
        amp = (0.02 if c < 3 else 1.5e5) * scale
        for _ in range(4):
            kv = 2.0 * math.pi / rng.uniform(8.0, 30.0)
            u = rng.standard_normal(3)
            u = kv * u / np.linalg.norm(u)
            ph = rng.uniform(0.0, 2.0 * math.pi)
            yz = (u[1] * j)[None, :] + (u[2] * k)[:, None] + ph
            w[c, 3:-3, 3:-3, 3:-3] += (0.5 * amp) * (torch.cos(yz)[:, :, None] * (fade * torch.cos(u[0] * i)) -
                                                      torch.sin(yz)[:, :, None] * (fade * torch.sin(u[0] * i)))
    return w


def _load_waves(case, core, w):
    """Restarts the core from a checkpoint in device memory that holds w:
    a saved state begins with the wavefield [9][nz][ny][row], rows padded to
    32 floats. Returns (checkpoint, its wavefield)."""
    buf = torch.zeros(core.state_bytes(), dtype=torch.uint8, device=DEV)
    torch.cuda.synchronize()
    core.save_state(dev_ptr=buf.data_ptr())
    f = _wave_of(case, buf)
    f.copy_(w)
    torch.cuda.synchronize()
    core.load_state(dev_ptr=buf.data_ptr())
    return buf


def _wave_of(case, buf):
    nz, ny, nx = case["nk"] + 6, case["nj"] + 6, case["ni"] + 6
    row = (nx + 31) // 32 * 32
    return buf[:9 * nz * ny * row * 4].view(torch.float32).view(9, nz, ny, row)[..., :nx]


class State:
    pass


def prepare(case, seed):
    s = State()
    s.case = case
    sc, fields = _scenario(case, seed)
    st = model.Setup(sc)
    nt, ns = case["steps"], case["nscen"]
    s.sta = _stations(case, seed)
    if ns == 1:
        s.core = model.Core(st)
        s.start = _load_waves(case, s.core, _waves(case, seed))
        if case["kind"] == "forward":
            s.core.set_stations(s.sta, 64)
            s.chk, s.start = s.start, None
    else:
        s.core = model.Batch(st, [(None if q == 0 else fields[q], 10 ** 8) for q in range(ns)])
        if ns * case["ni"] * case["nj"] * case["nk"] <= 8e6:
            for q in range(ns):
                w = _waves(case, seed + q).cpu().numpy()
                L.check(s.core.lib, s.core.lib.cgfd_batch_write_wavefield(s.core.handle, q, L.ptr(w)))
        if case["kind"] == "batch":
            s.core.set_stations(s.sta, 64)
    if case["kind"].endswith("adjoint"):
        rng = np.random.default_rng(seed + 5)
        s.target = 0.01 * rng.standard_normal((len(s.sta), nt, 9)).astype(np.float32)
        s.weight = np.array([1.0] * 3 + [1e-7] * 6, np.float32)
        s.target[:, :, 3:] *= 1e7
    st.close()
    for a in ("x", "y", "z", "lam", "mu", "rho"):  # the setup copied them
        setattr(sc, a, None)
    torch.cuda.synchronize()
    return s


# ---------------------------------------------------------------------------
# one pass


def _fault_out(f):
    return {"traction": f[0:3], "rate": f[3:6], "slip": f[6:9], "peak": f[9], "onset": f[10]}


def _split(v, axis=0):
    """Velocities and stresses apart."""
    return [v[:3], v[3:]] if axis == 0 else [v[..., :3], v[..., 3:]]


def _forward(s):
    c, core = s.case, s.core
    core.run(c["steps"])
    out = {"fault": [_fault_out(core.read_fault(q)) for q in range(c["faults"])]}
    if not c["buried"]:
        out["pg"] = core.read_pg()
    if c["out"] == "state":
        core.save_state(dev_ptr=s.chk.data_ptr())
        out["wave"] = _split(_wave_of(c, s.chk))
        out["stations"] = _split(core.read_stations(), -1)
    else:
        x = (_x_index(c) or [c["ni"] // 2])[0] + 3
        out["slices"] = [_split(core.read_slice(a, i)) for a, i in ((0, x), (1, c["nj"] // 2 + 3), (2, c["nk"] + 2))]
    return out


def _snapshot(bat, q, case):
    """Every fourth node of scenario q in each direction, velocity and stress."""
    n = [(case[a] + 3) // 4 for a in ("ni", "nj", "nk")]
    box = np.array([3, n[0], 4, 3, n[1], 4, 3, n[2], 4], np.int32)
    out = np.empty((9, n[2], n[1], n[0]), np.float32)
    L.check(bat.lib, bat.lib.cgfd_batch_read_snapshot(bat.handle, q, L.ptr(box), C.c_int(3), L.ptr(out)))
    return out


def _batch(s):
    c, bat = s.case, s.core
    bat.run(c["steps"])
    out = {"tractions": [], "slips": [], "snap_v": [], "snap_t": [], "sta": [], "pg": []}
    for q in range(c["nscen"]):
        f = bat.read_fault(q)
        v = _snapshot(bat, q, c)
        out["tractions"].append(f[0:3])
        out["slips"].append(f[3:10])
        out["snap_v"].append(v[:3])
        out["snap_t"].append(v[3:])
        out["sta"].append(bat.read_stations(q)[..., :3])
        if not c["buried"]:
            out["pg"].append(bat.read_pg(q))
    return {k: np.stack(v) for k, v in out.items() if v}


def _adjoint(s):
    c, core = s.case, s.core
    nt = c["steps"]
    core.load_state(dev_ptr=s.start.data_ptr())
    core.set_stations(s.sta, nt)
    core.adjoint_forward(nt)
    core.run(nt)
    tr = core.read_stations()
    r = (tr - s.target) * s.weight
    out = {"traces": _split(tr, -1)}
    if c["faults"]:
        g, gf = core.adjoint_fault(r)
        out["grad"] = _split(g)
        out["grad_fault"] = [gf[:, q] for q in range(7)]
    else:
        out["grad"] = _split(core.adjoint_initial(r))
    return out


def _batch_adjoint(s):
    c, bat = s.case, s.core
    nt = c["steps"]
    bat.set_stations(s.sta, nt)
    bat.adjoint_forward(nt)
    bat.run(nt)
    out = {"traces": [], "grad": [], "grad_fault": []}
    for q in range(c["nscen"]):
        tr = bat.read_stations(q)
        g, gf = bat.adjoint_fault(q, (tr - s.target) * s.weight)
        out["traces"].append(_split(tr, -1))
        out["grad"].append(_split(g))
        out["grad_fault"].append(gf)
    return {"traces": out["traces"], "grad": out["grad"], "grad_fault": [np.stack([f[:, p] for f in out["grad_fault"]])
                                                                          for p in range(7)]}


def run(state):
    return {"forward": _forward, "batch": _batch, "adjoint": _adjoint,
            "batch_adjoint": _batch_adjoint}[state.case["kind"]](state)


# ---------------------------------------------------------------------------
# the waves in 64 bits, from the published scheme: MacCormack-type 5-point
# one-sided operators whose direction alternates with the stage, RK4, CFS-PML
# with auxiliary variables, traction imaging and a reduced-order velocity
# gradient at the free surface

_CF = (-0.291647047, -0.666745142, 1.250117713, -0.333411808, 0.041686285)  # taps -1..3
_PAIRS = ((0, 0, 0), (1, 1, 0), (1, 1, 1), (0, 0, 1), (0, 1, 0), (1, 0, 0), (1, 0, 1), (0, 1, 1))
_SYM = ((3, 8, 7), (8, 4, 6), (7, 6, 5))  # components of the stress tensor


def _d(f, axis, fwd):
    """The one-sided operator at the physical points of the last three
    (ghost-inclusive) dimensions; axis 0 = x, 1 = y, 2 = z."""
    dim = f.dim() - 1 - axis
    out = None
    for t, cf in enumerate(_CF):
        o = t - 1 if fwd else 1 - t
        ix = [slice(None)] * (f.dim() - 3) + [slice(3, -3)] * 3
        n = f.shape[dim] - 6
        ix[dim] = slice(3 + o, 3 + o + n)
        v = (cf if fwd else -cf) * f[tuple(ix)]
        out = v if out is None else out + v
    return out


def _odd_ghosts(a):
    """Linear extrapolation of the coordinates into three ghost points per side."""
    for dim in (2, 1, 0):
        n = a.shape[dim]
        lo = [2 * a.narrow(dim, 0, 1) - a.narrow(dim, m, 1) for m in (3, 2, 1)]
        hi = [2 * a.narrow(dim, n - 1, 1) - a.narrow(dim, n - 1 - m, 1) for m in (1, 2, 3)]
        a = torch.cat(lo + [a] + hi, dim)
    return a


class _Exact:
    def __init__(self, case, seed):
        self.c = case
        ni, nj, nk = case["ni"], case["nj"], case["nk"]
        rng = np.random.default_rng(seed)
        x, y, z, topo = _grid(case, rng)
        lam, mu, rho = (t.double() for t in _media(case, z, topo, seed))
        self.xyz = [_odd_ghosts(t.double()) for t in (x, y, z)]

        def centre(a, axis):
            dim, s = 2 - axis, 0.0
            for o, w in ((-3, -0.01666667), (-2, 0.15), (-1, -0.75), (1, 0.75), (2, -0.15), (3, 0.01666667)):
                ix = [slice(3, -3)] * 3
                ix[dim] = slice(3 + o, a.shape[dim] - 3 + o)
                s = s + w * a[tuple(ix)]
            return s
        v = [torch.stack([centre(a, ax) for a in self.xyz]) for ax in range(3)]
        cr = [torch.linalg.cross(v[(d + 1) % 3], v[(d + 2) % 3], dim=0) for d in range(3)]
        self.jac = (cr[2] * v[2]).sum(0)
        self.m = [q / self.jac for q in cr]  # m[d][a]: derivative of the d-th curvilinear coordinate along a
        self.lam, self.mu, self.slw, self.l2m = lam, mu, 1.0 / rho, lam + 2.0 * mu
        self.dt, self.free = _dt(case), not case["buried"]
        self.faces = []
        for dim in range(3):
            for side in range(2):
                nl = _layers(case)[dim][side]
                if nl:
                    self.faces.append(self.face(dim, side, nl))
        if self.free:
            t = [q[:, -1] for q in self.m]  # (3, nj, ni) on the surface
            l, m = self.lam[-1], self.mu[-1]

            def dm(a, b):
                s = (a * b).sum(0)
                return torch.stack([torch.stack([l * a[p] * b[q] + m * a[q] * b[p] + (m * s if p == q else 0.0)
                                                 for q in range(3)], -1) for p in range(3)], -2)
            inv = torch.linalg.inv(dm(t[2], t[2]))
            self.mx, self.my = -inv @ dm(t[2], t[0]), -inv @ dm(t[2], t[1])

    def face(self, dim, side, nl):
        c = self.c
        n = (c["ni"], c["nj"], c["nk"])[dim]
        sl = [slice(None)] * 3  # (k, j, i)
        sl[2 - dim] = slice(0, nl + 1) if side == 0 else slice(n - nl - 1, n)
        d = [a[3:-3, 3:-3, 3:-3][tuple(sl)].diff(dim=2 - dim) for a in self.xyz]
        dh = float(torch.sqrt(d[0] ** 2 + d[1] ** 2 + d[2] ** 2).mean())
        r = 10.0 ** (-((math.log10(nl) - 1.0) / math.log10(2.0) + 4.0))
        u = torch.arange(nl + 1, dtype=torch.float64, device=DEV) / nl
        D, A, B = -3.0 * 7000.0 / (2.0 * dh * nl) * math.log(r) * u ** 2, 3.14 * (1.0 - u), 1.0 + u ** 2
        D = D / B
        A, B = A + D, 1.0 / B
        if side == 0:
            A, B, D = A.flip(0), B.flip(0), D.flip(0)
        sh = [1, 1, 1]
        sh[2 - dim] = nl + 1
        return dim, tuple(sl), A.view(sh), B.view(sh), D.view(sh)

    def momentum(self, d, g):
        """The rhs's part from the derivatives d (9 fields) along direction g."""
        e = self.m[g]
        v = [self.slw * sum(e[a] * d[_SYM[c][a]] for a in range(3)) for c in range(3)]
        return torch.stack(v + self.hooke([[e[a] * d[c] for a in range(3)] for c in range(3)]))

    def hooke(self, g):
        """Stress rates of the velocity gradient g[c][a]."""
        tr = g[0][0] + g[1][1] + g[2][2]
        return [self.lam * tr + 2.0 * self.mu * g[a][a] for a in range(3)] + [
            self.mu * (g[a][b] + g[b][a]) for a, b in ((1, 2), (0, 2), (0, 1))]

    def rhs(self, w, aux, dirs):
        d = [_d(w, ax, dirs[ax]) for ax in range(3)]
        part = [self.momentum(d[g], g) for g in range(3)]
        h = part[0] + part[1] + part[2]
        if self.free:
            h = torch.cat([h[:, :-4], self.surface(w, d, h[:, -4:], dirs)], 1)
        ar = []
        add = torch.zeros_like(h)
        for (dim, sl, A, B, D), a in zip(self.faces, aux):
            ix = (slice(None),) + sl
            r = part[dim][ix]
            if self.free and dim < 2:
                q = torch.einsum("jirc,cji->rji", self.mx if dim == 0 else self.my, d[dim][:3, -1])
                z = self.m[2][:, -1]
                s = [t[-1] for t in (self.lam, self.mu)]
                tr = z[0] * q[0] + z[1] * q[1] + z[2] * q[2]
                e = torch.stack([torch.zeros_like(tr)] * 3 + [s[0] * tr + 2.0 * s[1] * z[a] * q[a] for a in range(3)] +
                                [s[1] * (z[b] * q[a] + z[a] * q[b]) for a, b in ((1, 2), (0, 2), (0, 1))])
                r = torch.cat([r[:, :-1], r[:, -1:] + e[(slice(None),) + sl[1:]][:, None]], 1)
            add = add.index_put(_grid_ix(add, ix), (B - 1.0) * r - B * a, accumulate=True)
            ar.append(D * r - A * a)
        return h + add, ar

    def surface(self, w, d, h, dirs):
        """The top four layers' rhs: traction images in the momentum, reduced
        order for the vertical derivative of the velocity."""
        n = 4 if dirs[2] else 2
        v, t = h[:3], h[3:]
        out = []
        for c in range(3):
            T = [w[_SYM[c][a]][3:-3, 3:-3, 3:-3] for a in range(3)]
            con = [self.jac * sum(self.m[g][a] * T[a] for a in range(3)) for g in range(3)]
            pad = torch.nn.functional.pad
            z = torch.cat([con[2][:-1], torch.zeros_like(con[2][:1]), -con[2][-4:-1].flip(0)])
            z = pad(z, (3, 3, 3, 3, 3, 0))
            s = _d(pad(con[0], (3,) * 6), 0, dirs[0]) + _d(pad(con[1], (3,) * 6), 1, dirs[1]) + _d(z, 2, dirs[2])
            out.append(torch.cat([v[c][:4 - n], (s * self.slw / self.jac)[-n:]]))
        V = w[:3]
        ph = V[:, :, 3:-3, 3:-3]
        top = ph.shape[1] - 4  # the surface plane among the ghost-inclusive ones
        p = lambda o: ph[:, top + o]  # noqa: E731
        if dirs[2]:
            z1 = p(0) - p(-1)
            z2 = -7.0 / 6.0 * p(-2) + 8.0 / 6.0 * p(-1) - 1.0 / 6.0 * p(0)
        else:
            z1 = p(-1) - p(-2)
            z2 = 7.0 / 6.0 * p(-2) - 8.0 / 6.0 * p(-3) + 1.0 / 6.0 * p(-4)
        dx, dy = d[0][:3, -3:], d[1][:3, -3:]
        z0 = torch.einsum("jirc,cji->rji", self.mx, dx[:, 2]) + torch.einsum("jirc,cji->rji", self.my, dy[:, 2])
        dz = torch.stack([z2, z1, z0], 1)
        keep = self.lam, self.mu
        self.lam, self.mu = self.lam[-3:], self.mu[-3:]
        e = [q[:, -3:] for q in self.m]
        g = [[e[0][a] * dx[c] + e[1][a] * dy[c] + e[2][a] * dz[c] for a in range(3)] for c in range(3)]
        s = torch.stack(self.hooke(g))
        self.lam, self.mu = keep
        return torch.cat([torch.stack(out), torch.cat([t[:, :1], s], 1)])

    def step(self, w, aux, it):
        full = lambda h: torch.nn.functional.pad(h, (3,) * 6)  # noqa: E731
        cur, cura, end, enda = w, aux, w, aux
        for s in range(4):
            h, ar = self.rhs(cur, cura, [(q + s) % 2 for q in _PAIRS[it % 8]])
            h = full(h)
            b = self.dt * (1.0 / 6.0, 1.0 / 3.0, 1.0 / 3.0, 1.0 / 6.0)[s]
            end, enda = end + b * h, [x + b * y for x, y in zip(enda, ar)]
            if s < 3:
                a = self.dt * (0.5, 0.5, 1.0)[s]
                cur, cura = w + a * h, [x + a * y for x, y in zip(aux, ar)]
        return end, enda

    def start_aux(self):
        one = torch.zeros((9, self.c["nk"], self.c["nj"], self.c["ni"]), dtype=torch.float64, device=DEV)
        return [torch.zeros_like(one[(slice(None),) + f[1]]) for f in self.faces]

    def traces(self, w, sta):
        i, j, k = (torch.as_tensor(sta[:, q].astype(np.int64), device=DEV) for q in range(3))
        return w[:, k, j, i].T


def _grid_ix(a, ix):
    r = [torch.arange(n, device=a.device)[s] for n, s in zip(a.shape, ix)]
    return tuple(t.view([-1 if q == p else 1 for q in range(4)]) for p, t in enumerate(r))


def exact(case, seed):
    if case["faults"] or case["nscen"] > 1 or case["ni"] * case["nj"] * case["nk"] * case["steps"] > 2e7:
        return None
    if case["kind"] == "adjoint" and case["ni"] * case["nj"] * case["nk"] * case["steps"] > 2e6:
        return None
    e = _Exact(case, seed)
    sta = _stations(case, seed)
    w = _waves(case, seed).double()
    if case["kind"] == "adjoint":
        w.requires_grad_(True)
    w0, aux, tr, pg, dis = w, e.start_aux(), [], None, 0.0
    for it in range(case["steps"]):
        tr.append(e.traces(w, sta))
        old = w
        if case["kind"] == "adjoint":
            w, aux = e.step(w, aux, it)
            continue
        with torch.no_grad():
            w, aux = e.step(w, aux, it)
            v, v0 = w[:3, -4, 3:-3, 3:-3], old[:3, -4, 3:-3, 3:-3]
            acc, dis = (v - v0).abs() / e.dt, dis + 0.5 * (v + v0) * e.dt
            now = torch.cat([torch.stack([(q * q).sum(0).sqrt(), (q[:2] ** 2).sum(0).sqrt()] + list(q.abs()))
                             for q in (v, acc, dis)])
            pg = now if pg is None else torch.maximum(pg, now)
    tr = torch.stack(tr, 1)
    if case["kind"] == "adjoint":
        rng = np.random.default_rng(seed + 5)
        target = 0.01 * rng.standard_normal(tuple(tr.shape)).astype(np.float32)
        target[:, :, 3:] *= 1e7
        weight = torch.tensor([1.0] * 3 + [1e-7] * 6, dtype=torch.float64, device=DEV)
        r = (tr.detach() - torch.as_tensor(target, device=DEV).double()) * weight
        g, = torch.autograd.grad((tr * r).sum(), w0)
        ph = torch.zeros_like(g)
        ph[:, 3:-3, 3:-3, 3:-3] = g[:, 3:-3, 3:-3, 3:-3]
        return {"traces": _split(tr.detach(), -1), "grad": _split(ph)}
    pad = torch.nn.functional.pad
    out = {"fault": []}
    if not case["buried"]:
        out["pg"] = pad(pg, (3, 3, 3, 3))
    if case["out"] == "state":
        out["wave"] = _split(w)
        out["stations"] = _split(tr, -1)
    else:
        ph = w[:, 3:-3, 3:-3, 3:-3]
        out["slices"] = [_split(q) for q in (ph[..., case["ni"] // 2], ph[:, :, case["nj"] // 2], ph[:, -1])]
    return out
