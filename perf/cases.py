"""Workloads of the immersed-boundary library through its Python binding, with
the sizes its configurations use, their inputs, one pass of each, and what a
pass computes in plain FP64.

Lengths of a case are in um (the library's unit is 10 um); a box with walls
has them in y and is periodic in x and z.  A case is a dict with a "kind":

  couple     forces at the cells' sample sites spread onto the MAC grid, and
             velocities interpolated back to their data sites
  surface    RBF evaluation of cells at their sample sites (one matrix product
             per operator)
  channel    direct Helmholtz solves of the three velocity components and the
             pressure Poisson solve of a walled channel
  multigrid  one multigrid solve on a periodic box
  flow       advection, divergence and pressure gradient on the MAC grid
  boxes      many small periodic boxes: spread, interpolation, Helmholtz solve
  step       whole timesteps of a channel with cells, replayed as a graph
"""
import importlib.util
import math
import os
import sys

import numpy as np
import torch

ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))
UM = 0.1                                    # library length unit = 10 um
NU, RHO, DT = 10.0, 1e-3, 1e-4              # water, 0.1 us steps (library units)
WALL = 0.1                                  # moving wall, 1e-3 m/s
RBC_RADIUS = 3.91 * UM
PLT_RADII = (1.55 * UM, 0.50 * UM, 1.55 * UM)
INFLATE = 1.01                              # cells start inflated against their undeformed shapes


def _ibm():
    """The library's binding (the package's folder name is no identifier)."""
    if "ibm" not in sys.modules:
        spec = importlib.util.spec_from_file_location("ibm", os.path.join(ROOT, "ib.cu_amd", "ibm.py"))
        sys.modules["ibm"] = importlib.util.module_from_spec(spec)
        spec.loader.exec_module(sys.modules["ibm"])
    return sys.modules["ibm"]


def listed():
    return [
        # The smallest coupling: one sphere of 2562 markers in a periodic box
        # of 32 cells; launches and latency count.
        {"name": "couple_sphere", "kind": "couple", "lx": 16.0, "ly": 16.0, "lz": 16.0, "refinement": 32,
         "walls": False, "delta": "cosine", "rbc": 0, "plt": 0, "spheres": 1, "ns_rbc": 0, "nd_rbc": 0,
         "ns_plt": 2562, "nd_plt": 2562},
        # A middling suspension in a periodic box of 100 cells an axis (no
        # power of two, no whole number of 8-cell bricks), Peskin's kernel.
        {"name": "couple_ragged", "kind": "couple", "lx": 25.0, "ly": 25.0, "lz": 25.0, "refinement": 100,
         "walls": False, "delta": "peskin", "rbc": 18, "plt": 11, "spheres": 0, "ns_rbc": 8832, "nd_rbc": 2210,
         "ns_plt": 1552, "nd_plt": 605},
        # The benchmark's channel and suspension: 2,387,200 sample sites,
        # 684,000 data sites, 128 x 256 x 128 cells.
        {"name": "couple_suspension", "kind": "couple", "lx": 32.0, "ly": 64.0, "lz": 32.0, "refinement": 128,
         "walls": True, "delta": "cosine", "rbc": 200, "plt": 400, "spheres": 0, "ns_rbc": 8832, "nd_rbc": 2210,
         "ns_plt": 1552, "nd_plt": 605},
        # A few cells: positions and tangents of eight RBCs, FP64.
        {"name": "surface_few", "kind": "surface", "nd": 2210, "ns": 8832, "degree": 5, "cells": 8, "ops": 3,
         "precision": "f64"},
        # FP32 products for callers that need no more: 64 RBCs (192 columns).
        {"name": "surface_single", "kind": "surface", "nd": 2210, "ns": 8832, "degree": 5, "cells": 64, "ops": 3,
         "precision": "f32"},
        # The benchmark's RBCs: positions, tangents and second derivatives of
        # 200 cells (the membrane models need all six), FP64.
        {"name": "surface_suspension", "kind": "surface", "nd": 2210, "ns": 8832, "degree": 5, "cells": 200,
         "ops": 6, "precision": "f64"},
        # The benchmark's channel: one step's four linear systems.
        {"name": "channel_solves", "kind": "channel", "lx": 32.0, "ly": 64.0, "lz": 32.0, "refinement": 128},
        # A pressure Poisson solve of a periodic box of 96 cells an axis, FP32
        # V-cycles in FP64 defect correction.
        {"name": "multigrid_box", "kind": "multigrid", "n": 96, "precision": 32, "poisson": True},
        # The explicit fluid operators on a ragged channel, 90 x 180 x 90 cells.
        {"name": "flow_ragged", "kind": "flow", "lx": 32.0, "ly": 64.0, "lz": 32.0, "refinement": 90, "walls": True},
        # 64 independent periodic boxes of 32 cells an axis with up to 20 cells each.
        {"name": "boxes_batch", "kind": "boxes", "boxes": 64, "n": 32, "most": 20, "ns": 546},
        # A small channel: eight RBCs on 64 cells an axis.
        {"name": "step_channel", "kind": "step", "lx": 16.0, "ly": 16.0, "lz": 16.0, "refinement": 64, "rbc": 8,
         "plt": 0, "ns_rbc": 8832, "nd_rbc": 2210, "ns_plt": 1552, "nd_plt": 605},
        # The benchmark's whole timestep.
        {"name": "step_suspension", "kind": "step", "lx": 32.0, "ly": 64.0, "lz": 32.0, "refinement": 128, "rbc": 200,
         "plt": 400, "ns_rbc": 8832, "nd_rbc": 2210, "ns_plt": 1552, "nd_plt": 605},
    ]


def _log_uniform(rng, lo, hi):
    return int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))


def draw(rng):
    kind = rng.choice(["couple", "couple", "surface", "surface", "channel", "multigrid", "flow", "boxes", "step"])
    if kind == "couple":
        l = float(rng.choice([16, 24, 32]))
        tall = rng.choice([1.0, 2.0])
        slots = int(l // 8) ** 2 * max(1, int(l * tall / 4.5))
        return {"kind": kind, "lx": l, "ly": l * tall, "lz": l, "refinement": _log_uniform(rng, 32, 128 if l == 32 else 110),
                "walls": rng.random() < 0.6, "delta": rng.choice(["cosine", "cosine", "peskin", "bspline3"]),
                "rbc": _log_uniform(rng, 1, slots), "plt": rng.choice([0, _log_uniform(rng, 1, 2 * slots)]), "spheres": 0,
                "ns_rbc": _log_uniform(rng, 500, 8832), "nd_rbc": _log_uniform(rng, 300, 2210),
                "ns_plt": _log_uniform(rng, 200, 1552), "nd_plt": _log_uniform(rng, 100, 605)}
    if kind == "surface":
        nd = _log_uniform(rng, 300, 2210)
        return {"kind": kind, "nd": nd, "ns": _log_uniform(rng, nd, 4 * nd), "degree": rng.choice([0, 5]),
                "cells": _log_uniform(rng, 1, 200), "ops": rng.choice([1, 3, 6]),
                "precision": rng.choice(["f64", "f64", "f64", "f32", "bf16x3"])}
    if kind == "channel":
        r = rng.choice([32, 64, 128])
        return {"kind": kind, "lx": 16.0, "ly": rng.choice([8.0, 16.0, 32.0, 48.0]), "lz": rng.choice([8.0, 16.0]),
                "refinement": r // 2}
    if kind == "multigrid":
        return {"kind": kind, "n": 8 * rng.randint(3, 12), "precision": rng.choice([32, 64]),
                "poisson": rng.random() < 0.5}
    if kind == "flow":
        tall = rng.choice([1.0, 2.0])
        return {"kind": kind, "lx": 32.0, "ly": 32.0 * tall, "lz": 32.0, "refinement": _log_uniform(rng, 24, 96),
                "walls": rng.random() < 0.6}
    if kind == "boxes":
        return {"kind": kind, "boxes": _log_uniform(rng, 1, 64), "n": rng.choice([16, 24, 32]),
                "most": rng.randint(1, 20), "ns": _log_uniform(rng, 200, 546)}
    l = rng.choice([16.0, 32.0])
    rbc = rng.randint(1, 4 if l == 16.0 else 48)
    return {"kind": kind, "lx": l, "ly": l, "lz": l, "refinement": rng.choice([32, 64]), "rbc": rbc,
            "plt": rng.choice([0, rng.randint(1, 40)]), "ns_rbc": _log_uniform(rng, 1200, 4000),
            "nd_rbc": _log_uniform(rng, 300, 1000), "ns_plt": _log_uniform(rng, 500, 1552),
            "nd_plt": _log_uniform(rng, 150, 400)}


# ----------------------------------------------------------------------
# Sites, cells and fields
# ----------------------------------------------------------------------
def _spiral(n, device):
    """(theta, phi) of the n-point Bauer spiral on the sphere."""
    z = -1.0 + (2.0 * torch.arange(n, dtype=torch.float64, device=device) + 1.0) / n
    phi = torch.asin(z)
    return torch.stack([torch.remainder(math.sqrt(math.pi * n) * phi, 2 * math.pi), phi])


def _unit(params):
    t, p = params
    return torch.stack([torch.cos(t) * torch.cos(p), torch.sin(t) * torch.cos(p), torch.sin(p)])


def _shape(which, params):
    """Undeformed RBC (biconcave), platelet (ellipsoid) or sphere, 3 x n."""
    x, y, z = _unit(params)
    if which == "rbc":
        r2 = x * x + y * y
        return RBC_RADIUS * torch.stack([x, 0.5 * z * (0.21 + 2.0 * r2 - 1.12 * r2 * r2), y])
    if which == "plt":
        return torch.stack([PLT_RADII[0] * x, PLT_RADII[1] * y, PLT_RADII[2] * z])
    return RBC_RADIUS * torch.stack([x, y, z])


def _poses(case, seed):
    """Centres (um) and spin / tilt angles of the RBCs (layers of 8 um slots,
    discs normal to y) and the platelets (5 um slots between the layers)."""
    rng = np.random.default_rng(seed)
    lx, ly, lz = case["lx"], case["ly"], case["lz"]

    def lattice(count, pitch):
        """Centres on x-z slots, and each one's layer."""
        nx, nz = max(1, int(lx // pitch)), max(1, int(lz // pitch))
        layer, slot = np.divmod(np.arange(count), nx * nz)
        return np.stack([(slot % nx + 0.5) * lx / nx, 0.0 * slot, (slot // nx + 0.5) * lz / nz], axis=1), layer

    rc, layer = lattice(case["rbc"], 8.0)
    layers = int(layer.max()) + 1 if len(layer) else 0
    rc[:, 1] = (layer + 0.5) * ly / max(layers, 1)
    pc, layer = lattice(case["plt"], 5.0)
    pc[:, 1] = (layer % (layers - 1) + 1) * ly / layers if layers > 1 else (0.15 if layers else 0.5) * ly
    rc += (rng.random(rc.shape) - 0.5) * np.array([0.08, 0.1, 0.08])
    pc += (rng.random(pc.shape) - 0.5) * np.array([0.5, 0.0, 0.5])
    angles = lambda n, tilt: np.stack([2 * math.pi * rng.random(n), math.radians(tilt) * (rng.random(n) - 0.5)], axis=1)  # noqa: E731
    return (rc, angles(len(rc), 2.0)), (pc, angles(len(pc), 0.0))


def _posed(points, pose, device):
    """Copies (3, cells, n) of points (3, n): spun about y, tilted about x, moved."""
    centres = torch.from_numpy(pose[0] * UM).to(device)
    a = torch.from_numpy(pose[1]).to(device)
    cs, sn, ct, st = torch.cos(a[:, :1]), torch.sin(a[:, :1]), torch.cos(a[:, 1:]), torch.sin(a[:, 1:])
    x = cs * points[0] + sn * points[2]
    z = -sn * points[0] + cs * points[2]
    y = ct * points[1] - st * z
    z = st * points[1] + ct * z
    return torch.stack([x, y, z]) + centres.T[:, :, None]


def _generator(seed, device):
    g = torch.Generator(device=device)
    g.manual_seed(int(seed))
    return g


def _domain(ibm, case, walls):
    l = [case["lx"] * UM, case["ly"] * UM, case["lz"] * UM]
    return [ibm.periodic(l[0]), ibm.dirichlet(l[1]) if walls else ibm.periodic(l[1]), ibm.periodic(l[2])]


def _mesh(case, walls):
    """Mesh width, and per component and axis (points, cells, wall, shift) of
    the MAC grid: points of a component lie at (i + shift) h."""
    l = [case["lx"], case["ly"], case["lz"]]
    unit = l[0]
    for v in l[1:]:
        a, b = max(unit, v), min(unit, v)
        while b > 1e-9:
            a, b = b, a % b if a % b > 1e-9 and b - a % b > 1e-9 else 0.0
        unit = a
    h = unit * UM / case["refinement"]
    cells = [int(round(v * UM / h)) for v in l]
    axes = []
    for c in range(4):                       # three components, then the cell centres
        row = []
        for j in range(3):
            wall = walls and j == 1
            row.append((cells[j] - 1 if wall and c == j else cells[j], cells[j], wall,
                        (1.0 if wall else 0.0) if c == j else 0.5))
        axes.append(row)
    return h, axes


def _fields(axes, count, seed, device):
    """Smooth flow plus noise on the first `count` component grids, as flat
    x-fastest vectors."""
    g = _generator(seed, device)
    out = []
    for c in range(count):
        n = [axes[c][j][0] for j in range(3)]
        k = [torch.arange(n[j], dtype=torch.float64, device=device) * (2 * math.pi / n[j]) for j in range(3)]
        ph = torch.rand(3, generator=g, dtype=torch.float64, device=device) * 6.0
        f = (torch.sin(k[2] + ph[2])[:, None, None] * torch.cos(2 * k[1] + ph[1])[None, :, None]
             + torch.cos(k[0] + ph[0])[None, None, :])
        f = f + 0.1 * torch.randn(f.shape, generator=g, dtype=torch.float64, device=device)
        out.append((0.1 * f).reshape(-1).contiguous())
    return out


# ----------------------------------------------------------------------
# RBF operators of the surfaces (inputs of "surface")
# ----------------------------------------------------------------------
def _basis(sample, data, degree, kind):
    """The r^7 splines of the chord distance and the monomials of the unit
    sphere at the sample sites, or their derivatives in (theta, phi): rows
    (nd + terms), columns ns."""
    ts, ps = sample[:, None, :]
    td, pd = data[:, :, None]
    c, s = torch.cos(ts - td), torch.sin(ts - td)
    cps, sps, cpd, spd = torch.cos(ps), torch.sin(ps), torch.cos(pd), torch.sin(pd)
    t = c * cps * cpd + sps * spd
    r = torch.sqrt((2.0 * (1.0 - t)).clamp_min(0.0))
    dt = {"t": -s * cps * cpd, "p": -c * sps * cpd + cps * spd}
    d2 = {"tt": -c * cps * cpd, "tp": s * sps * cpd, "pp": -t}
    if kind == "":
        phi = r ** 7
    elif len(kind) == 1:
        phi = -7.0 * r ** 5 * dt[kind]
    else:
        phi = 35.0 * r ** 3 * dt[kind[0]] * dt[kind[1]] - 7.0 * r ** 5 * d2[kind]
    # monomials x^a y^b z^e, e <= 1, differentiated through the sphere's map
    t, p = sample
    x = _unit(sample)
    first = {"t": torch.stack([-x[1], x[0], torch.zeros_like(t)]),
             "p": torch.stack([-torch.cos(t) * torch.sin(p), -torch.sin(t) * torch.sin(p), torch.cos(p)])}
    second = {"tt": torch.stack([-x[0], -x[1], torch.zeros_like(t)]),
              "tp": torch.stack([torch.sin(t) * torch.sin(p), -torch.cos(t) * torch.sin(p), torch.zeros_like(t)]),
              "pp": -x}
    rows = []
    for e in (0, 1):
        for tot in range(e, degree + 1):
            for a in range(tot - e, -1, -1):
                powers = (a, tot - e - a, e)

                def mono(wrt):
                    left, coef = list(powers), 1.0
                    for i in wrt:
                        coef *= left[i]
                        left[i] -= 1
                    if coef == 0:
                        return torch.zeros_like(t)
                    v = torch.full_like(t, coef)
                    for i in range(3):
                        for _ in range(left[i]):
                            v = v * x[i]
                    return v
                if kind == "":
                    v = mono(())
                elif len(kind) == 1:
                    v = sum(mono((i,)) * first[kind][i] for i in range(3))
                else:
                    v = sum(mono((i,)) * second[kind][i] for i in range(3))
                    for i in range(3):
                        for j in range(3):
                            v = v + mono((i, j)) * first[kind[0]][i] * first[kind[1]][j]
                rows.append(v)
    return torch.cat([phi, torch.stack(rows)])


KINDS = ("", "t", "p", "tt", "tp", "pp")


def _operators(case, device):
    """Evaluator and derivative matrices, sample-major (ns, nd + terms)."""
    data, sample = _spiral(case["nd"], device), _spiral(case["ns"], device)
    terms = (case["degree"] + 1) ** 2
    a = _basis(data, data, case["degree"], "")
    m = torch.zeros((case["nd"] + terms,) * 2, dtype=torch.float64, device=device)
    m[:, :case["nd"]] = a
    m[:case["nd"], case["nd"]:] = a[case["nd"]:].T
    lu, piv = torch.linalg.lu_factor(m)
    return [torch.cat([torch.linalg.lu_solve(lu, piv, b).T for b in
                       _basis(sample, data, case["degree"], k).split(512, dim=1)]).contiguous()
            for k in KINDS[:case["ops"]]]


def _surface_sites(case, seed, device):
    """Data sites of the cells, rows comp * cells + cell."""
    pose = {"lx": 32.0, "ly": 64.0, "lz": 32.0, "rbc": case["cells"], "plt": 0}
    x = _posed(INFLATE * _shape("rbc", _spiral(case["nd"], device)), _poses(pose, seed)[0], device)
    return x.reshape(3 * case["cells"], case["nd"]).contiguous()


# ----------------------------------------------------------------------
# Markers of "couple" and "boxes"
# ----------------------------------------------------------------------
def _markers(case, seed, device):
    """Sample and data sites (lists of SoA vectors, one per cell type) and
    forces at the sample sites."""
    rbc, plt = _poses(case, seed)
    xs, xd, fs = [], [], []
    g = _generator(seed, device)
    kinds = [("rbc", rbc, case["ns_rbc"], case["nd_rbc"]), ("plt", plt, case["ns_plt"], case["nd_plt"])]
    if case["spheres"]:
        rng = np.random.default_rng(seed)
        centre = np.array([[case["lx"], case["ly"], case["lz"]]]) / 2 + rng.random((case["spheres"], 3)) - 0.5
        kinds = [("sphere", (centre, np.zeros((case["spheres"], 2))), case["ns_plt"], case["nd_plt"])]
    for which, pose, ns, nd in kinds:
        if len(pose[0]) == 0:
            continue
        for n, to in ((ns, xs), (nd, xd)):
            to.append(_posed(INFLATE * _shape(which, _spiral(n, device)), pose, device).reshape(-1).contiguous())
        fs.append(torch.randn(xs[-1].numel(), generator=g, dtype=torch.float64, device=device))
    return xs, xd, fs


def _box_markers(case, seed, device):
    """Box-local positions (3, n), box offsets and forces: up to `most` cells
    a box at the slots of a jittered 3 x 3 x 3 lattice."""
    rng, count = np.random.default_rng(seed), np.random.default_rng(case["most"])   # sizes are the case's own
    spacing = 32.0 * UM / 3
    shapes = [_shape("rbc", _spiral(case["ns"], "cpu")).numpy(),
              _shape("plt", _spiral(max(case["ns"] * 7 // 10, 1), "cpu")).numpy()]
    pts, offsets = [], [0]
    for _ in range(case["boxes"]):
        n = 0
        for k in range(int(count.integers(1, case["most"] + 1))):
            ref = shapes[int(count.integers(2))]
            q, r = np.linalg.qr(rng.standard_normal((3, 3)))
            slot = np.array([k % 3, k // 3 % 3, k // 9])
            pts.append(q @ ref + ((slot + 0.5 + 0.1 * (rng.random(3) - 0.5)) * spacing)[:, None])
            n += ref.shape[1]
        offsets.append(offsets[-1] + n)
    x = torch.from_numpy(np.ascontiguousarray(np.concatenate(pts, axis=1))).to(device)
    f = torch.randn(x.numel(), generator=_generator(seed, device), dtype=torch.float64, device=device)
    return x, offsets, f


# ----------------------------------------------------------------------
# prepare
# ----------------------------------------------------------------------
_held = {}


def _context():
    """One context for the operators (as a program holds one per thread)."""
    if "ctx" not in _held:
        _held["ctx"] = _ibm().Context(0)
    return _held["ctx"]


def _step_context():
    """Captured steps need a stream of their own."""
    if "step" not in _held:
        _held["stream"] = torch.cuda.Stream()
        _held["step"] = _ibm().Context(0, stream=_held["stream"])
    return _held["step"], _held["stream"]


def prepare(case, seed):
    ibm, kind, dev = _ibm(), case["kind"], torch.device("cuda", 0)
    s = {"kind": kind}
    if kind == "step":
        return _prepare_step(case, seed)
    ctx = s["ctx"] = _context()
    if kind == "couple":
        s["grids"] = ibm.mac_grids(_domain(ibm, case, case["walls"]), case["refinement"])
        _, axes = _mesh(case, case["walls"])
        s["xs"], s["xd"], s["fs"] = _markers(case, seed, dev)
        s["u"] = _fields(axes, 3, seed, dev)
        s["delta"] = case["delta"]
        s["fe"] = [torch.empty_like(u) for u in s["u"]]
        s["ul"] = [torch.empty_like(x) for x in s["xd"]]
    elif kind == "surface":
        mats = _operators(case, dev)
        s["op"] = ibm.RbfOperator(ctx, case["precision"], mats, case["nd"])
        del mats
        s["x"] = _surface_sites(case, seed, dev)
        s["y"] = torch.empty((case["ops"], 3 * case["cells"], case["ns"]), dtype=torch.float64, device=dev)
    elif kind == "channel":
        domain = _domain(ibm, case, True)
        grids = list(ibm.mac_grids(domain, case["refinement"]))
        neumann = [domain[0], ibm.neumann(case["ly"] * UM), domain[2]]
        grids.append(ibm.centered_grid(neumann, case["refinement"]))
        s["solvers"] = [ibm.FftSolver(ctx, g) for g in grids]
        s["ops"] = [(1.0, -DT * NU / 2)] * 3 + [(0.0, 1.0)]
        _, axes = _mesh(case, True)
        s["b"] = _fields(axes, 4, seed, dev)
        s["x"] = [torch.empty_like(b) for b in s["b"]]
    elif kind == "multigrid":
        grid = ibm.centered_grid([ibm.periodic(16 * UM)] * 3, case["n"])
        s["mg"] = ibm.Multigrid(ctx, grid, (0.0, 1.0) if case["poisson"] else (1.0, -DT * NU / 2), case["precision"])
        s["b"] = _box_field(case, seed, dev)
        s["x"] = torch.empty_like(s["b"])
    elif kind == "flow":
        domain = _domain(ibm, case, case["walls"])
        s["grids"] = ibm.mac_grids(domain, case["refinement"])
        s["pgrid"] = ibm.centered_grid([domain[0], ibm.neumann(case["ly"] * UM) if case["walls"] else domain[1],
                                        domain[2]], case["refinement"])
        _, axes = _mesh(case, case["walls"])
        *s["u"], s["p"] = _fields(axes, 4, seed, dev)
        s["h"] = [torch.empty_like(u) for u in s["u"]]
        s["g"] = [torch.zeros_like(u) for u in s["u"]]
        s["d"] = torch.empty_like(s["p"])
    elif kind == "boxes":
        s["grids"] = ibm.mac_grids([ibm.periodic(32 * UM)] * 3, case["n"])
        x, s["offsets"], s["f"] = _box_markers(case, seed, dev)
        s["x"] = x.reshape(-1).contiguous()
        size = case["boxes"] * case["n"] ** 3
        g = _generator(seed + 1, dev)
        s["u"] = [torch.randn(size, generator=g, dtype=torch.float64, device=dev) for _ in range(3)]
        s["fe"] = [torch.empty(size, dtype=torch.float64, device=dev) for _ in range(3)]
        s["ul"] = torch.empty_like(s["x"])
        s["v"] = torch.empty(size, dtype=torch.float64, device=dev)
        s["mg"] = ibm.BoxesMultigrid(ctx, s["grids"][0], case["boxes"], (1.0, -DT * NU))
    return s


def _box_field(case, seed, dev):
    n = case["n"]
    b = _fields([[(n, n, False, 0.5)] * 3], 1, seed, dev)[0]
    return b - b.mean() if case["poisson"] else b


def _prepare_step(case, seed):
    """A channel with cells whose membranes resist tension and bending, some
    steps in, and its step captured."""
    ibm, dev = _ibm(), torch.device("cuda", 0)
    ctx, stream = _step_context()
    rbc, plt = _poses(case, seed)
    cells, sites = [], []
    with torch.cuda.stream(stream):
        for which, pose, nd, ns, degree, membrane in (
                ("rbc", rbc, case["nd_rbc"], case["ns_rbc"], 5, ("skalak", 2.5e-3, 2.5e-1, 2e-6, False)),
                ("plt", plt, case["nd_plt"], case["ns_plt"], 0, ("neohookean", 1e-1, 1.0, 2e-5, True))):
            if len(pose[0]) == 0:
                continue
            data, sample = _spiral(nd, dev), _spiral(ns, dev)
            ops = ibm.rbf_build(ctx, data, sample, degree, ("value", "t", "p", "tt", "tp", "pp"))
            dops = ibm.rbf_build(ctx, data, data, degree, ("t", "p", "tt", "tp", "pp"))
            ref = _shape(which, data)
            cells.append({"ops": ibm.RbfOperator(ctx, "f64", ops, nd), "data_ops": ibm.RbfOperator(ctx, "f64", dops, nd),
                          "cells": len(pose[0]), "weights": ibm.sphere_weights(ctx, sample),
                          "membrane": ibm.membrane(*membrane), "reference": ref.reshape(-1).contiguous()})
            sites.append(_posed(INFLATE * ref, pose, dev).reshape(-1).contiguous())
            del ops, dops
        solver = ibm.Solver(ctx, _domain(ibm, case, True), case["refinement"], DT, NU, density=RHO, tolerance=1e-10,
                            max_iterations=60, cell_types=cells)
        grids, _ = solver.grids()
        ub = [torch.zeros(grids[i].size, dtype=torch.float64, device=dev) for i in range(3)]
        ibm.boundary_apply(ctx, grids[0], 1, 1, ub[0], value=WALL, order=2)
        state = solver.zero_state(sites)
        for _ in range(2):
            solver.step(state, boundary=ub)
        solver.capture(state, boundary=ub)
        stream.synchronize()
    return {"kind": "step", "solver": solver, "state": state, "ub": ub}


# ----------------------------------------------------------------------
# run
# ----------------------------------------------------------------------
def run(s):
    ibm, kind, ctx = _ibm(), s["kind"], s.get("ctx")
    if kind == "couple":
        ibm.spread_sets(ctx, s["grids"], s["delta"], s["xs"], s["fs"], out=s["fe"])
        ibm.interpolate_sets(ctx, s["grids"], s["delta"], s["xd"], s["u"], outs=s["ul"])
        return {"fe": s["fe"], "ul": s["ul"]}
    if kind == "surface":
        return ibm.rbf_eval(ctx, [s["op"]], [s["x"]], ys=[s["y"]])
    if kind == "channel":
        return [p.solve(b, op, x=x) for p, b, op, x in zip(s["solvers"], s["b"], s["ops"], s["x"])]
    if kind == "multigrid":
        return s["mg"].solve(s["b"], rtol=1e-10, x=s["x"])[0]
    if kind == "flow":
        ibm.advection(ctx, s["grids"], s["u"], out=s["h"])
        ibm.divergence(ctx, s["grids"], s["u"], out=s["d"])
        ibm.gradient(ctx, s["pgrid"], s["p"], out=s["g"])
        return {"h": s["h"], "d": s["d"], "g": s["g"]}
    if kind == "boxes":
        ibm.spread_boxes(ctx, s["grids"], "cosine", s["offsets"], s["x"], s["f"], out=s["fe"])
        ibm.interpolate_boxes(ctx, s["grids"], "cosine", s["offsets"], s["x"], s["u"], out=s["ul"])
        s["mg"].solve(s["u"][0], x=s["v"], rtol=1e-10)
        return {"fe": s["fe"], "ul": s["ul"], "v": s["v"]}
    s["solver"].replay(s["state"])
    st = s["state"]
    return {"u": st.u, "p": st.p, "x": st.xs}


# ----------------------------------------------------------------------
# work
# ----------------------------------------------------------------------
def _points(case, walls, count):
    _, axes = _mesh(case, walls)
    return [math.prod(axes[c][j][0] for j in range(3)) for c in range(count)]


def _solve_work(n, points):
    """A direct solve: vector read and written; two transforms each way of
    every axis and the tridiagonal sweeps."""
    return {"bytes": 16.0 * points, "flops": points * (5.0 * math.log2(max(n, 2)) * 2 + 20.0)}


def _marker_work(ns, nd, points):
    return {"bytes": 48.0 * ns + 8.0 * points + 48.0 * nd + 8.0 * min(points, 3 * 64 * nd),
            "flops": (ns + nd) * 3 * (64 * 3 + 60.0)}


def work(case):
    kind = case["kind"]
    if kind == "couple":
        n_small = case["spheres"] or case["plt"]
        ns = case["rbc"] * case["ns_rbc"] + n_small * case["ns_plt"]
        nd = case["rbc"] * case["nd_rbc"] + n_small * case["nd_plt"]
        return _marker_work(ns, nd, sum(_points(case, case["walls"], 3)))
    if kind == "surface":
        n = 3 * case["cells"]
        size = {"f64": 8, "f32": 4, "bf16x3": 4}[case["precision"]]
        return {"bytes": case["ops"] * (case["ns"] * case["nd"] * float(size) + 8.0 * case["ns"] * n)
                + 8.0 * n * case["nd"], "flops": 2.0 * case["ops"] * case["ns"] * case["nd"] * n}
    if kind == "channel":
        p = _points(case, True, 4)
        w = [_solve_work(max(case["refinement"], 2) ** 2, v) for v in p]
        return {k: sum(x[k] for x in w) for k in ("bytes", "flops")}
    if kind == "multigrid":
        # a vector read and one written; about ten V-cycles of two degree-4
        # smoothings, a residual and the transfers
        p = float(case["n"]) ** 3
        return {"bytes": 16.0 * p, "flops": 10 * 100.0 * p}
    if kind == "flow":
        p = _points(case, case["walls"], 4)
        return {"bytes": 8.0 * (3 * sum(p[:3]) + 2 * p[3]), "flops": 40.0 * sum(p)}
    if kind == "boxes":
        p = 3.0 * case["boxes"] * case["n"] ** 3
        m = case["boxes"] * (case["most"] + 1) / 2 * case["ns"] * 0.85
        w = _marker_work(m, m, p)
        return {"bytes": w["bytes"] + 16.0 * p / 3, "flops": w["flops"] + 6 * 100.0 * p / 3}
    flops = bytes_ = ns = nd = 0.0
    for c, d, m in ((case["rbc"], case["nd_rbc"], case["ns_rbc"]), (case["plt"], case["nd_plt"], case["ns_plt"])):
        if c:
            flops += 2.0 * d * (6 * m * 3 * c + 5 * d * 3 * c + 5 * m * c)
            bytes_ += 8.0 * (6 * m * d + 5 * d * d) + 8.0 * 6 * c * d
            ns, nd = ns + c * m, nd + c * d
    p = _points(case, True, 4)
    w = _marker_work(ns, nd, sum(p[:3]))
    # velocities and pressure read and written once
    return {"bytes": bytes_ + w["bytes"] + 16.0 * sum(p), "flops": flops + w["flops"] + 150.0 * sum(p)}


# ----------------------------------------------------------------------
# exact: plain FP64 torch, without the library
# ----------------------------------------------------------------------
def _phi(delta, r):
    a = r.abs()
    if delta == "cosine":
        v = 0.25 * (1.0 + torch.cos(0.5 * math.pi * r))
    elif delta == "peskin":
        near = (3 - 2 * a + torch.sqrt((1 + 4 * a - 4 * a * a).clamp_min(0.0))) / 8
        far = (5 - 2 * a - torch.sqrt((-7 + 12 * a - 4 * a * a).clamp_min(0.0))) / 8
        v = torch.where(a < 1, near, far)
    else:
        near = 2.0 / 3 - a * a + a ** 3 / 2
        far = (2 - a) ** 3 / 6
        v = torch.where(a < 1, near, far)
    return torch.where(a < 2, v, torch.zeros_like(v))


def _stencil(axis, h, x, delta):
    """Per marker the four grid indices along an axis (wrapped, or clamped at
    walls), the weights, and at walls whether each index is on the grid."""
    u = x / h - axis[3]
    i = torch.floor(u)[None, :] + torch.arange(-1, 3, device=x.device, dtype=torch.float64)[:, None]
    w = _phi(delta, i - u[None, :])
    i = i.long()
    if axis[2]:
        return i.clamp(0, axis[0] - 1), w, (i >= 0) & (i < axis[0])
    return torch.remainder(i, axis[1]), w, None


def _exact_couple(axes, h, delta, x, f, xd, u):
    """fe from (x, f), (3, n) each, and ul of the fields u at xd."""
    fe, ul = [], []
    for c in range(3):
        n = [axes[c][j][0] for j in range(3)]
        fe.append(torch.zeros(n[0] * n[1] * n[2], dtype=torch.float64, device=x.device))
        for spread, pos in ((True, x), (False, xd)):
            ix, w, ok = zip(*[_stencil(axes[c][j], h, pos[j], delta) for j in range(3)])
            got = torch.zeros(pos.shape[1], dtype=torch.float64, device=x.device)
            for a in range(4):
                for b in range(4):
                    for d in range(4):
                        at = ix[0][d] + n[0] * (ix[1][b] + n[1] * ix[2][a])
                        v = w[0][d] * w[1][b] * w[2][a]
                        if spread:
                            if ok[1] is not None:
                                v = v * ok[1][b]
                            fe[c].index_add_(0, at, v * f[c] * h ** -3)
                        else:
                            got += v * u[c][at]
            if not spread:
                ul.append(got)
    return fe, ul


def _modes(n, h, device):
    """Orthonormal eigenvectors (columns) and eigenvalues of the periodic
    three-point Laplacian on n points."""
    i = torch.arange(n, dtype=torch.float64, device=device)
    q, lam = [], []
    for k in range(n // 2 + 1):
        a = 2 * math.pi / n * torch.remainder(k * i, n)
        for v in (torch.cos(a), torch.sin(a)) if 0 < 2 * k < n else (torch.cos(a),):
            q.append(v / v.norm())
            lam.append(-4.0 / (h * h) * math.sin(math.pi * k / n) ** 2)
    return torch.stack(q, 1), torch.tensor(lam, dtype=torch.float64, device=device)


def _along(a, q, d):
    """a with dimension d multiplied by q."""
    return (a.movedim(d, -1).contiguous().reshape(-1, q.shape[0]) @ q).reshape(
        [a.shape[k] for k in range(a.dim()) if k != d % a.dim()] + [q.shape[1]]).movedim(-1, d)


def _exact_periodic_solve(b, n, h, sigma, tau):
    """(sigma + tau L) x = b on periodic n^3 boxes; mean-free if singular."""
    q, lam = _modes(n, h, b.device)
    d = sigma + tau * (lam[:, None, None] + lam[None, :, None] + lam[None, None, :])
    s = b.reshape(-1, n, n, n)
    for k in (1, 2, 3):
        s = _along(s, q, k)
    if sigma == 0.0:
        d[0, 0, 0] = 1.0
        s[:, 0, 0, 0] = 0.0
    s = s / d
    for k in (1, 2, 3):
        s = _along(s, q.T, k)
    return s.reshape(-1)


def _exact_channel_solve(b, axes, h, sigma, tau, neumann, face):
    """(sigma I2 + tau L) x = b, periodic in x and z, walls in y: one
    tridiagonal system per mode."""
    nx, ny, nz = (axes[j][0] for j in range(3))
    (qx, lx), (qz, lz) = _modes(nx, h, b.device), _modes(nz, h, b.device)
    lam = lz[:, None] + lx[None, :]
    s = _along(_along(b.reshape(nz, ny, nx), qx, 2), qz, 0).movedim(1, 0).contiguous()
    ident = torch.ones(ny, dtype=torch.float64)
    diag = torch.full((ny,), -2.0, dtype=torch.float64)
    if neumann:
        diag[0] += 1.0
        diag[-1] += 1.0
    elif not face:
        diag[0] -= 1.0
        diag[-1] -= 1.0
        ident[0] = ident[-1] = 0.75
    off = tau / (h * h)
    singular = sigma == 0.0 and neumann
    if singular:
        s[:, 0, 0] -= s[:, 0, 0].mean()
    cp, dp = [], []
    for j in range(ny):
        m = ident[j].item() * (sigma + tau * lam) + off * diag[j].item()
        lower, right = off, s[j]
        if singular and j == ny - 1:
            right = right.clone()
            lower = torch.full_like(m, off)
            m[0, 0], right[0, 0], lower[0, 0] = 1.0, 0.0, 0.0
        den = m - lower * cp[-1] if cp else m
        cp.append(off / den)
        dp.append((right - lower * dp[-1]) / den if dp else right / den)
    x = [dp[-1]]
    for j in range(ny - 2, -1, -1):
        x.append(dp[j] - cp[j] * x[-1])
    x = torch.stack(x[::-1])
    if singular:
        x[:, 0, 0] -= x[:, 0, 0].mean()
    return _along(_along(x.movedim(0, 1), qx.T, 2), qz.T, 0).contiguous().reshape(-1)


def _exact_flow(axes, h, u, p, walls):
    """Advection, divergence and gradient by shifted copies; fields are
    [z, y, x], the wall faces of v are kept as zero rows."""
    dims = {0: 2, 1: 1, 2: 0}
    v = [a.reshape([axes[c][j][0] for j in (2, 1, 0)]) for c, a in enumerate(u)]
    pc = p.reshape([axes[3][j][0] for j in (2, 1, 0)])

    def ends(a, axis, lo, hi):
        """Face values between the points of a centred field; walls in y get
        ghost points of lo / hi times the end rows."""
        d = dims[axis]
        if walls and axis == 1:
            return torch.cat([lo * a.narrow(d, 0, 1), a, hi * a.narrow(d, a.shape[d] - 1, 1)], d)
        return torch.cat([a.narrow(d, a.shape[d] - 1, 1), a], d)

    def to_face(a, axis, avg, ghost=-1.0):
        d, e = dims[axis], ends(a, axis, ghost, ghost)
        n = e.shape[d] - 1
        lo, hi = e.narrow(d, 0, n), e.narrow(d, 1, n)
        return (lo + hi) / 2 if avg else (hi - lo) / h

    def to_centre(a, axis, avg, faces=False):
        """From faces; v's vector holds the interior faces, an averaged one (faces) the wall faces too."""
        d = dims[axis]
        if walls and axis == 1:
            if not faces:
                z = torch.zeros_like(a.narrow(d, 0, 1))
                a = torch.cat([z, a, z], d)
            n = a.shape[d] - 1
            lo, hi = a.narrow(d, 0, n), a.narrow(d, 1, n)
        else:
            lo, hi = a, torch.roll(a, -1, d)
        return (lo + hi) / 2 if avg else (hi - lo) / h

    def inner(a, axis):
        """Interior faces of a face field with the wall faces."""
        return a.narrow(dims[axis], 1, a.shape[dims[axis]] - 2) if walls and axis == 1 else a

    def padded(a, axis):
        if walls and axis == 1:
            z = torch.zeros_like(a.narrow(dims[axis], 0, 1))
            return torch.cat([z, a, z], dims[axis])
        return a

    h_out = []
    for i in range(3):
        total = None
        for j in range(3):
            if i == j:
                a = to_centre(v[i], i, True)
                t = inner(to_face(a * a, i, False), i)
            else:
                # u_j averaged along i and u_i averaged along j, on the edges
                a = to_face(padded(v[j], j) if j == 1 else v[j], i, True)
                b = to_face(padded(v[i], i) if i == 1 else v[i], j, True)
                t = to_centre(a * b, j, False, faces=True)
                t = inner(t, i) if i == 1 else t
            total = t if total is None else total + t
        h_out.append(total.reshape(-1).contiguous())
    div = sum(to_centre(v[i], i, False) for i in range(3))
    grad = [inner(to_face(pc, i, False, 1.0), i).reshape(-1).contiguous() for i in range(3)]
    return {"h": h_out, "d": div.reshape(-1).contiguous(), "g": grad}


def exact(case, seed):
    kind, dev = case["kind"], torch.device("cuda", 0)
    if kind == "couple":
        h, axes = _mesh(case, case["walls"])
        xs, xd, fs = _markers(case, seed, dev)
        u = _fields(axes, 3, seed, dev)
        cat = lambda v: torch.cat([a.reshape(3, -1) for a in v], 1)  # noqa: E731
        fe, ul = _exact_couple(axes, h, case["delta"], cat(xs), cat(fs), cat(xd), u)
        ul = torch.stack(ul).split([a.numel() // 3 for a in xd], dim=1)
        return {"fe": fe, "ul": [a.reshape(-1).contiguous() for a in ul]}
    if kind == "surface":
        x = _surface_sites(case, seed, dev)
        return [torch.stack([x @ m[:, :case["nd"]].T for m in _operators(case, dev)])]
    if kind == "channel":
        h, axes = _mesh(case, True)
        b = _fields(axes, 4, seed, dev)
        return [_exact_channel_solve(b[c], axes[c], h, *((1.0, -DT * NU / 2) if c < 3 else (0.0, 1.0)), c == 3, c == 1)
                for c in range(4)]
    if kind == "multigrid":
        b = _box_field(case, seed, dev)
        return _exact_periodic_solve(b, case["n"], 16 * UM / case["n"],
                                     *((0.0, 1.0) if case["poisson"] else (1.0, -DT * NU / 2)))
    if kind == "flow":
        h, axes = _mesh(case, case["walls"])
        *u, p = _fields(axes, 4, seed, dev)
        return _exact_flow(axes, h, u, p, case["walls"])
    if kind == "boxes":
        n, h = case["n"], 32 * UM / case["n"]
        x, offsets, f = _box_markers(case, seed, dev)
        g = _generator(seed + 1, dev)
        u = [torch.randn(case["boxes"] * n ** 3, generator=g, dtype=torch.float64, device=dev) for _ in range(3)]
        f = f.reshape(3, -1)
        fe, ul = [[] for _ in range(3)], []
        axes = [[(n, n, False, 0.0 if c == j else 0.5) for j in range(3)] for c in range(3)]
        for b in range(case["boxes"]):
            part = slice(offsets[b], offsets[b + 1])
            ub = [v[b * n ** 3:(b + 1) * n ** 3] for v in u]
            a, w = _exact_couple(axes, h, "cosine", x[:, part], f[:, part], x[:, part], ub)
            for c in range(3):
                fe[c].append(a[c])
            ul.append(torch.stack(w))
        return {"fe": [torch.cat(v) for v in fe], "ul": torch.cat(ul, 1).reshape(-1),
                "v": _exact_periodic_solve(u[0], n, h, 1.0, -DT * NU)}
    return None
