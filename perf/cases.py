"""Cases that time the framework as its users call it, with their reference results.

The framework is a narrow-band FLIP solver on two basins: the dense `FlipBasin` and the
two-resolution `SparseBasin`. A program steps a basin (`step`), or runs the phases of a
step by itself: particles to grid, the pressure projection, grid to particles, and the
adjoints of the three. The cases cover both basins from 60 cm cells (the smallest grids
of the tests, where launches and latency count) to 15 cm dense and 5 cm sparse (the sizes
of the benchmark), the solve in each storage precision (`precision` 0 FP32, 1 FP16, 2
BF16), and the forward and the backward direction.

`prepare` builds a basin, starts the balanced vortex and moves it off balance from the
seed (its waves, or its particles' places and velocities). `exact` restates the phases in FP64 with torch on dense index grids.
"""
import math
import os
import sys

import numpy as np
import torch

ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))
sys.path.insert(0, os.path.join(ROOT, "maelstrom.jl_amd"))
import maelstrom_amd as mael  # noqa: E402
from maelstrom_amd import dense, sparse  # noqa: E402

AX = ("U", "V", "W")
VN = ("VX", "VY", "VZ")
CN = tuple("C%d" % k for k in range(9))
SOLID, LIQUID, AIR = 0, 1, 2
F64 = torch.float64


# ── the cases ────────────────────────────────────────────────────────────────

def _case(name, basin, path, dx, radius=18.0, depth=12.0, precision=0, tol=1e-6):
    return {"name": name, "basin": basin, "path": path, "dx": dx, "radius": radius, "depth": depth,
            "precision": precision, "tol": tol}


def listed():
    return [
        # one particles-to-grid and grid-to-particles pair on the tests' 64x64x32 grid: a
        # coarse preview or a fit's inner loop, where each call's launches count
        _case("dense_transfers_60cm", "dense", "transfers", 0.6),
        # the same on the benchmark's 256x256x128 grid
        _case("dense_transfers_15cm", "dense", "transfers", 0.15),
        # one pressure solve from a cold start on the small grid, at the default tolerance
        _case("dense_project_60cm", "dense", "project", 0.6, tol=1e-4),
        # a whole step of the dense benchmark
        _case("dense_step_15cm", "dense", "step", 0.15),
        # the gradient of one step's transfers and projection (the three adjoints), 128x128x64
        _case("dense_backward_30cm", "dense", "backward", 0.3),
        # the sparse transfers alone at the benchmark's resolution, where they move most
        _case("sparse_p2g_5cm", "sparse", "p2g", 0.05),
        _case("sparse_g2p_5cm", "sparse", "g2p", 0.05),
        # the default FP32 solve of a stirred surface at a preview's resolution
        _case("sparse_project_20cm", "sparse", "project", 0.2, tol=5e-4),
        # the benchmark's mixed-precision solve to 1e-6
        _case("sparse_project_5cm_fp16", "sparse", "project", 0.05, precision=1),
        # the adjoints on the sparse basin, between preview and final resolution
        _case("sparse_backward_15cm", "sparse", "backward", 0.15, precision=2),
        # whole steps: the tests' smallest sparse basin, and the benchmark's headline
        _case("sparse_step_60cm", "sparse", "step", 0.6, tol=5e-4),
        _case("sparse_step_5cm_fp16", "sparse", "step", 0.05, precision=1),
    ]


def draw(rng):
    """A case of the same ranges: any path, resolution (over its logarithm), basin and solve."""
    basin = rng.choice(("dense", "sparse"))
    lo = 0.15 if basin == "dense" else 0.05
    dx = round(math.exp(rng.uniform(math.log(lo), math.log(0.6))), 4)
    if basin == "dense":
        path = rng.choice(("transfers", "project", "step", "backward"))
        precision, tol = 0, rng.choice((1e-4, 1e-6))
    else:
        path = rng.choice(("p2g", "g2p", "project", "step", "backward"))
        precision = rng.choice((0, 1, 2))
        tol = 1e-6 if precision else 5e-4   # FP32 storage without FP64 refinement stalls near 1e-4
    if path == "backward":
        tol = 1e-6
        precision = 0 if basin == "dense" else rng.choice((1, 2))
        dx = max(dx, 0.15)
    c = _case("", basin, path, dx, round(rng.uniform(12.0, 18.0), 2), round(rng.uniform(8.0, 12.0), 2), precision, tol)
    del c["name"]
    return c


# ── a basin under way ────────────────────────────────────────────────────────

class _Buffer:
    """A device array of the library as torch takes it."""

    def __init__(self, ptr, count, dtype):
        self.__cuda_array_interface__ = {"shape": (count,), "typestr": np.dtype(dtype).str, "data": (ptr, False),
                                         "version": 2, "strides": None}


def _view(s, name, count=None):
    ptr, cnt, dt = s._info(name)
    t = torch.as_tensor(_Buffer(ptr, cnt if count is None else count, dt), device="cuda")
    t.basin = s   # the memory is the basin's, which lives as long as the view
    return t


def _solve(case):
    o = dict(tol=case["tol"])
    if case["basin"] == "sparse":
        o.update(maxiter=240, restart=20, policy=2, boost=1.5, precision=case["precision"])
    elif case["path"] == "backward":
        o.update(maxiter=200, refine=1)
    return o


def _dt(s, speed):
    """The time step of a 24 Hz frame cut to the basin's CFL number (the benchmark's rule)."""
    frame = 1.0 / 24
    return frame / math.ceil(frame / (s.cfl * s.grid.dx / max(speed, 1e-3)))


def _fine(s):
    """Names and live counts of the outputs' fine arrays."""
    return s.nslots * sparse.BCELLS, s.nslots * sparse.BFACES


def _make(case, seed):
    b = mael.Basin(radius=case["radius"], depth=case["depth"], Γ=225.0 * case["radius"] / 18.0, core=2.5)
    dx, area = case["dx"], (case["radius"] / 18.0) ** 2
    waves = mael.narutowaves(seed=int(seed) % (1 << 31))
    if case["basin"] == "dense":
        stir = mael.Stir(b, waves=waves, race=mael.Race(eddy=3.0))
        n = mael.flipgrid(b, dx).n
        s = mael.FlipBasin(b, dx, cfl=4.0, stir=stir, capacity=min(8 * n[0] * n[1] * n[2], 6_000_000))
        mael.initialize(s)
    else:
        stir = mael.Stir(b, waves=waves, race=mael.Race(eddy=3.0), surface=True)
        nb = mael.sparsegrid(b, dx).nb
        blocks = min(nb[0] * nb[1] * nb[2], int(12000 * (0.05 / dx) ** 2 * area) + 300)
        s = mael.SparseBasin(b, dx, stir=stir, cfl=4.0, blocks=blocks, capacity=2500 * blocks + 200_000)
        sparse.initialize(s)
    s.steps = int(seed) % 100_000
    return s


def _disturb(s, seed):
    """Particles under way: moved along their velocities by part of a step, each at its own
    time within it, their velocities and affine rows off the balanced flow."""
    s.sync()
    g = torch.Generator(device="cuda").manual_seed(int(seed))
    n, dx = s.n, s.grid.dx
    x = [_view(s, f, n) for f in ("PX", "PY", "PZ")]
    v = [_view(s, f, n) for f in VN]
    dt = _dt(s, float(max(t.abs().max() for t in v)))

    def normal():
        return torch.randn(n, generator=g, device="cuda")

    for a in range(3):
        v[a] += 0.1 * normal()
        x[a] += 0.5 * dt * v[a] + 0.05 * dx * normal()
    for f in CN:
        _view(s, f, n).add_(normal(), alpha=0.1)
    _view(s, "LAG", n).copy_((torch.rand(n, generator=g, device="cuda") - 0.5) * dt)
    torch.cuda.synchronize()
    return dt


def _flags(s, case, seed):
    """Valid-face flags as an extrapolation leaves them: set up to six cells above the
    surface, with a few faces it did not reach."""
    g = torch.Generator(device="cuda").manual_seed(int(seed) + 1)
    for a, ax in enumerate(AX):
        if case["basin"] == "dense":
            n1, n2, n3 = s.n_cells
            phi = _view(s, "PHI").view(n3, n2, n1)
            reach = torch.cat([phi, phi.narrow(2 - a, phi.shape[2 - a] - 1, 1)], 2 - a) < 6 * s.grid.dx
            f = _view(s, "F" + ax)
        else:
            nc, nf = _fine(s)
            phi = _view(s, "PHI_F", nc).view(-1, 16, 16, 16)
            reach = torch.cat([phi, phi.narrow(3 - a, 15, 1)], 3 - a) < 6 * s.grid.dx
            f = _view(s, "F%s_F" % ax, nf)
        f.copy_(reach.reshape(-1) & (torch.rand(f.numel(), generator=g, device="cuda") > 2e-4))
    torch.cuda.synchronize()


def prepare(case, seed):
    s = _make(case, seed)
    path = case["path"]
    m = dense if case["basin"] == "dense" else sparse
    st = {"case": case, "s": s, "solve": _solve(case)}
    if path == "step":
        st["dt"] = _dt(s, m.maxspeed(s))
        s.steps = 0
        return st
    dt = st["dt"] = _disturb(s, seed)
    if path == "project":
        # the state a step projects
        if m is dense:
            for phase in (dense.advect, dense.particles2grid):
                phase(s, dt)
            dense.redistance(s)
            dense.classify(s)
            dense.filltrapped(s)
            dense.forces(s, dt)
            for ax in AX:
                s.copy(ax + "0", ax)
        else:
            lib = mael.lib()
            s.ctx.check(lib.mael_sparse_advect(s.h, dt, 0, float(s.basin.g), int(s.steps)))
            sparse.particles2grid(s, dt)
            sparse.redistance(s)
            sparse.classify(s)
            s.ctx.check(lib.mael_sparse_filltrapped(s.h, 32))
            s.ctx.check(lib.mael_sparse_forces(s.h, dt, float(s.t), float(s.basin.g)))
            s.sync()
            st["u"] = [(_view(s, f), _view(s, f).clone()) for ax in AX for f in (ax + "_F", ax + "_C")]
            st["p"] = [_view(s, "P_F"), _view(s, "P_C")]
        st["gamma"] = m.gamma_for(s, dt)
    else:
        m.particles2grid(s, dt)
        s.sync()
        if path in ("transfers", "g2p"):
            _flags(s, case, seed)
    if path == "backward":
        m.classify(s)
        m.project(s, dt, **st["solve"])
        m.grid2particles(s, dt)
        s.sync()
        g = torch.Generator(device="cuda").manual_seed(int(seed) + 2)
        st["pb"] = [(_view(s, "PB_" + f, s.n), torch.randn(s.n, generator=g, device="cuda") * (1.0 if f in VN else 0.1))
                    for f in VN + CN]
    st["out"] = _outputs(s, case)
    s.sync()
    torch.cuda.synchronize()
    return st


def _outputs(s, case):
    """The arrays a pass of the case's path computes."""
    flat, path, n = case["basin"] == "dense", case["path"], s.n
    faces = AX if flat else tuple(ax + p for ax in AX for p in ("_F", "_C"))
    cells = {"PHI": ("PHI",) if flat else ("PHI_F", "PHI_C"), "P": ("P",) if flat else ("P_F", "P_C")}
    names = []
    if path in ("transfers", "p2g"):
        names += list(faces + cells["PHI"])
    if path in ("transfers", "g2p"):
        names += list(VN + CN)
    if path == "project":
        names += list(faces + cells["P"]) + ["F" + f for f in faces]
    if path == "backward":
        names += ["PB_" + f for f in VN + CN]
        names += ["UB0_" + f for f in faces]
    if path == "step":
        # the whole domain on the grid: on the sparse basin the coarse grid, which holds the
        # fine blocks' restriction under them (the order of the pool's slots is the
        # allocator's, and a block on the edge of a mark moves all that follow)
        names += list(AX) + ["PHI", "P"] if flat else [ax + "_C" for ax in AX] + ["PHI_C", "P_C"]
    out = {}
    for f in names:
        count = None
        if f in VN + CN or f.startswith("PB_"):
            count = n
        elif f.endswith("_F"):
            nc, nf = _fine(s)
            count = nc if f in ("PHI_F", "P_F") else nf
        out[f] = _view(s, f, count)
    return out


def run(state):
    s, case, dt, path = state["s"], state["case"], state["dt"], state["case"]["path"]
    m = dense if case["basin"] == "dense" else sparse
    if path == "step":
        m.step(s, dt, **state["solve"])
        return _outputs(s, case)   # the level set's two buffers change places within a step
    elif path == "transfers":
        m.particles2grid(s, dt)
        m.grid2particles(s, dt)
    elif path == "p2g":
        m.particles2grid(s, dt)
    elif path == "g2p":
        m.grid2particles(s, dt)
    elif path == "project":
        # a cold start: the pressure from zero and the velocity before the projection
        if case["basin"] == "dense":
            for ax in AX:
                s.copy(ax, ax + "0")
            m.project(s, dt, gamma=state["gamma"], warm=0, **state["solve"])
        else:
            for p in state["p"]:
                p.zero_()
            for u, u0 in state["u"]:
                u.copy_(u0)
            torch.cuda.current_stream().synchronize()   # torch's stream and the basin's are two
            m.project(s, dt, gamma=state["gamma"], **state["solve"])
    else:
        # a backward pass from this loss's cotangents
        s.sync()
        for pb, seed in state["pb"]:
            pb.copy_(seed)
        torch.cuda.current_stream().synchronize()
        m.grid2particles_adjoint(s, dt)
        m.project_adjoint(s, **state["solve"])
        m.particles2grid_adjoint(s, dt)
    return state["out"]


# ── what a pass cannot do without ────────────────────────────────────────────

def _sizes(case):
    """(particles, fine cells, coarse cells) expected: the band holds 8 particles a cell in
    four cells under the surface, live blocks follow it (counted at 5, 20 and 60 cm)."""
    dx, disc = case["dx"], math.pi * case["radius"] ** 2
    n = 8 * 4 * disc / dx ** 2
    if case["basin"] == "dense":
        side = 2 * (case["radius"] + 2 * dx) / dx
        return n, side * side * (case["depth"] + 3.0) / dx, 0
    coarse = (2 * case["radius"] / (4 * dx)) ** 2 * (case["depth"] + 3.0) / (4 * dx)
    fine = min(4096 * 13 * (case["radius"] / (16 * dx)) ** 2 + 64 * 4096, 64 * coarse)
    return n, fine, coarse


def work(case):
    """Bytes: each particle array and each grid array of the path read and written once (a
    solve's once an iteration). FP32 arrays, FP16 and BF16 ones in the V-cycle."""
    n, fine, coarse = _sizes(case)
    cells = fine + coarse
    p2g = 64 * n + cells * (3 * 8 + 8)            # a particle's 16 floats; u0 and u, φ0 and φ
    g2p = 60 * n + cells * 15                     # x, then v and the rows; u and its flags
    resample = 136 * n + 12 * cells
    e = 2 if case["precision"] else 4
    iteration = cells * ((5 * 3 + 8) * e + 36)    # the V-cycle's passes and CG's, each array once
    project = cells * 50 + 15 * iteration
    rest = cells * (7 * 9 + 24 + 30) + 80 * n     # redistance, advection, forces, extrapolation
    path = case["path"]
    halves = 2 if case["basin"] == "sparse" else 1
    by = {"transfers": p2g + g2p, "p2g": p2g, "g2p": g2p, "project": project, "backward": p2g + project + g2p,
          "step": halves * (p2g + g2p + resample + project + rest)}[path]
    transfer = n * 3 * 27 * 12
    fl = {"transfers": 2 * transfer, "p2g": transfer, "g2p": transfer, "project": 15 * 120 * cells,
          "backward": 2 * transfer + 15 * 120 * cells,
          "step": halves * (2 * transfer + (15 * 120 + 300) * cells)}[path]
    return {"bytes": float(by), "flops": float(fl)}


def tolerance(case):
    """About four times the distance from `exact` measured with FP32 rounding."""
    tol = case["tol"]
    return {"transfers": {"rel": 6e-5, "max": 1e-2}, "p2g": {"rel": 1e-4, "max": 0.1}, "g2p": {"rel": 5e-4, "max": 0.5},
            # a solve stops at its own relative residual
            "project": {"rel": 2 * tol + 1e-5, "max": 0.1, "differ": 1e-6},
            "backward": {"rel": 2 * tol + 3e-5, "max": 0.1},
            # two correct steps differ by their solves, and by what follows from the few
            # particles that those move over a cell's side
            "step": {"rel": 0.01, "max": 0.9}}[case["path"]]


# ── the phases in FP64 ───────────────────────────────────────────────────────

def exact(case, seed):
    """`run`'s outputs in FP64; None for whole steps, and for solves of over 3 M cells."""
    path = case["path"]
    if path == "step" or (path in ("project", "backward") and sum(_sizes(case)[1:]) > 1.2e7):
        return None
    st = prepare(case, seed)
    s, dt = st["s"], st["dt"]
    G = _Dense(s) if case["basin"] == "dense" else _Sparse(s)
    P = {f: _view(s, f, s.n).double() for f in ("PX", "PY", "PZ", "LAG") + VN + CN}
    out = {}
    if path in ("transfers", "p2g"):
        u0, phi0 = G.faces("%s0"), G.cells("PHI0")
        phi = G.union(P, dt, phi0)
        u = G.blend(*_deposit(G, P, dt), u0, phi)
        out.update(G.named("%s", u))
        out.update(G.named_cells("PHI", phi))
    if path in ("transfers", "g2p"):
        if path == "g2p":
            u = G.faces("%s")
        out.update(_gathered(G, P, u, G.faces("F%s"), dt, s.basin.g))
    if path == "project":
        u = G.faces("%s0") if case["basin"] == "dense" else G.faces("%s")
        u, p = _Poisson(G).project(u, st["gamma"], 0.1 * case["tol"])
        out.update(G.named("%s", u))
        out.update(G.named_cells("P", p))
        out.update(dict.fromkeys(["F" + f for f in out if f[0] != "P"]))   # flags have no FP64 value
    if path == "backward":
        pb = {f: t.double() for f, (_, t) in zip(VN + CN, st["pb"])}
        out.update(_backward(G, P, pb, dt, case["tol"]))
    torch.cuda.synchronize()
    return out


def _offset(axis, a):
    return 0.0 if axis == a else 0.5


def _nodes(q):
    """First node and the three quadratic B-spline weights along one axis."""
    b = torch.floor(q - 0.5)
    f = q - b
    return b.long(), (0.5 * (1.5 - f) ** 2, 0.75 - (f - 1.0) ** 2, 0.5 * (f - 0.5) ** 2)


def _stencil(G, P, a):
    """The 27 nodes of each particle on axis a's faces: (index, inside, weight, offsets in m)."""
    shape = G.face_shape(a)   # (z, y, x)
    q = [(P[f] - G.lo[k]) / G.dx - _offset(k, a) for k, f in enumerate(("PX", "PY", "PZ"))]
    bw = [_nodes(t) for t in q]
    for mz in range(3):
        for my in range(3):
            for mx in range(3):
                at = [bw[k][0] + m for k, m in enumerate((mx, my, mz))]
                w = bw[0][1][mx] * bw[1][1][my] * bw[2][1][mz]
                inside = torch.ones_like(at[0], dtype=torch.bool)
                lin = torch.zeros_like(at[0])
                for k in (2, 1, 0):
                    n = shape[2 - k]
                    inside &= (at[k] >= 0) & (at[k] < n)
                    lin = lin * n + at[k].clamp(0, n - 1)
                yield lin, inside, w, [(at[k].double() - q[k]) * G.dx for k in range(3)]


def _deposit(G, P, dt):
    """Momentum and weight on the faces of the whole (fine) grid, per axis."""
    r = (-P["LAG"] / dt).clamp(-0.5, 0.5) - 0.5
    wt = 35.0 / 16.0 * (1.0 - r * r) ** 3
    mom, wgt = [], []
    for a in range(3):
        N = math.prod(G.face_shape(a))
        m, w = torch.zeros(N, dtype=F64, device="cuda"), torch.zeros(N, dtype=F64, device="cuda")
        for lin, inside, c, d in _stencil(G, P, a):
            c = torch.where(inside, c * wt, 0.0)
            v = P[VN[a]] + sum(P[CN[3 * a + k]] * d[k] for k in range(3))
            m = m.index_add(0, lin, c * v) if m.requires_grad or v.requires_grad else m.index_add_(0, lin, c * v)
            w.index_add_(0, lin, c)
        mom.append(m)
        wgt.append(w)
    return mom, wgt


def _gather(G, P, a, whole, present):
    """(value, affine row) of a face field of the whole grid at the particles. Nodes off the
    grid read the nearest face on the dense basin and nothing on the sparse one."""
    val = torch.zeros_like(P["PX"])
    row = [torch.zeros_like(val) for _ in range(3)]
    for lin, inside, c, d in _stencil(G, P, a):
        if not G.clamps:
            c = torch.where(inside & present[lin], c, 0.0)
        t = c * whole[lin]
        val = val + t
        row = [r + t * e for r, e in zip(row, d)]
    return val, [4.0 / G.dx ** 2 * r for r in row]


def _reached(G, P, flags):
    ok = torch.ones(P["PX"].shape, dtype=torch.bool, device="cuda")
    for a in range(3):
        whole, present = G.whole(a, flags[a])
        ok &= _gather(G, P, a, whole, present)[0] > 0.999
    return ok


def _gathered(G, P, u, flags, dt, g):
    ok = _reached(G, P, flags)
    out = {}
    for a in range(3):
        whole, present = G.whole(a, u[a])
        val, row = _gather(G, P, a, whole, present)
        out[VN[a]] = torch.where(ok, val, P[VN[a]] - (g * dt if a == 2 else 0.0))
        for k in range(3):
            out[CN[3 * a + k]] = torch.where(ok, row[k], 0.0)
    return out


def _splat(G, P, dt):
    """Least distance of a particle's surface (a ball of half a cell, moved to where its
    speed carries it) to the fine cell centres round it."""
    v = [P[f] for f in VN]
    c = (torch.sqrt(v[0] ** 2 + v[1] ** 2 + v[2] ** 2) * dt / G.dx).clamp(0.0, 1.0)
    c = c * c * (3.0 - 2.0 * c)
    h = 0.25 * c * c
    ahead = h * (9.0 / 16 - h * (7.0 / 10 - h * 3.0 / 7)) / (27.0 / 64 + h * (3.0 / 16 - h * (3.0 / 20 + h / 7.0)))
    t = P["LAG"] + ahead * dt
    q = [(P[f] + t * v[k] - G.lo[k]) / G.dx for k, f in enumerate(("PX", "PY", "PZ"))]
    nz, ny, nx = G.cell_shape
    phi = torch.full((nz * ny * nx,), 1e30, dtype=F64, device="cuda")
    at = [torch.floor(t).long() for t in q]
    for dk in (-1, 0, 1):
        for dj in (-1, 0, 1):
            for di in (-1, 0, 1):
                i, j, k = at[0] + di, at[1] + dj, at[2] + dk
                ok = (i >= 0) & (i < nx) & (j >= 0) & (j < ny) & (k >= 0) & (k < nz)
                d = torch.sqrt(sum((c.double() + 0.5 - p) ** 2 for c, p in zip((i, j, k), q))) * G.dx - 0.5 * G.dx
                phi.scatter_reduce_(0, ((k * ny + j) * nx + i)[ok], d[ok], "amin")
    return phi


def _theta(a, b):
    return torch.nan_to_num(a / (a - b), nan=1.0).clamp(0.01, 1.0)   # 0 / 0 only where no row reads it


def _grid_faces(n, a):
    """(lower cell, upper cell, is the lower there, is the upper there) of the faces along a
    of a grid of n = (nx, ny, nz) cells."""
    K, J, I = torch.meshgrid(*[torch.arange(n[k] + (k == a), device="cuda") for k in (2, 1, 0)], indexing="ij")
    hi = [I, J, K]
    lo = [t - int(k == a) for k, t in enumerate(hi)]

    def lin(t):
        t = [x.clamp(0, n[k] - 1) for k, x in enumerate(t)]
        return ((t[2] * n[1] + t[1]) * n[0] + t[0]).reshape(-1)
    return lin(lo), lin(hi), (lo[a] >= 0).reshape(-1), (hi[a] < n[a]).reshape(-1)


class _Dense:
    """The dense basin's arrays as FP64 tensors; its own grid is the whole grid."""
    clamps = True

    def __init__(self, s):
        self.s, self.dx, self.lo = s, float(s.grid.dx), [float(x) for x in s.grid.lo]
        self.n = s.n_cells
        self.cell_shape = (self.n[2], self.n[1], self.n[0])

    def face_shape(self, a):
        return tuple(self.n[k] + (k == a) for k in (2, 1, 0))

    def faces(self, pattern):
        return [_view(self.s, pattern % ax).double() for ax in AX]

    def cells(self, name):
        return _view(self.s, name).double()

    def named(self, pattern, u):
        return {pattern % ax: t for ax, t in zip(AX, u)}

    def named_cells(self, name, t):
        return {name: t}

    def whole(self, a, u):
        return u, None

    def union(self, P, dt, phi0):
        return torch.minimum(phi0 + self.dx, _splat(self, P, dt))

    def face_phi(self, a, phi):
        lo, hi, has_lo, has_hi = _grid_faces(self.n, a)   # a face on the domain's side reads its one cell
        return 0.5 * (torch.where(has_lo, phi[lo], phi[hi]) + torch.where(has_hi, phi[hi], phi[lo]))

    def blend(self, mom, wt, u0, phi):
        full, deep = float(self.s.nmin), (self.s.band - 1) * self.dx
        return [torch.where(self.face_phi(a, phi) >= -deep,
                            (mom[a] + (full - wt[a]).clamp(min=0.0) * u0[a]) / wt[a].clamp(min=full), u0[a])
                for a in range(3)]


class _Sparse:
    """The sparse basin's arrays as FP64 tensors: a field is (fine pool, coarse grid), and
    the whole fine grid is the pool's values at their places on a dense grid."""
    clamps = False

    def __init__(self, s):
        self.s, self.dx, self.lo = s, float(s.grid.dx), [float(x) for x in s.grid.lo]
        self.nb = [int(x) for x in s.grid.nb]
        self.n, self.nc = [16 * x for x in self.nb], [4 * x for x in self.nb]
        self.cell_shape = (self.n[2], self.n[1], self.n[0])
        _, where, ns, _ = s.topology()
        self.where = torch.as_tensor(where[:ns].astype(np.int64), device="cuda")
        self.live = self.where[:, 0] >= 0
        self.ncell, self.nface = _fine(s)
        blocks = torch.zeros(self.nb[2], self.nb[1], self.nb[0], dtype=torch.bool, device="cuda")
        w = self.where[self.live]
        blocks[w[:, 2], w[:, 1], w[:, 0]] = True
        self.covered = blocks.repeat_interleave(4, 0).repeat_interleave(4, 1).repeat_interleave(4, 2).reshape(-1)
        c = self.coords(None)
        self.cell_at = self.place(c, self.cell_shape)   # the whole grid's index of each pool cell
        self.pool = torch.full((math.prod(self.cell_shape),), -1, dtype=torch.int32, device="cuda")
        ok = self.livemask(sparse.BCELLS)
        self.pool[self.cell_at[ok]] = torch.arange(self.ncell, device="cuda", dtype=torch.int32)[ok]

    def livemask(self, per):
        return self.live.repeat_interleave(per)

    def coords(self, a):
        """Global (I, J, K) of the pool's cells (a None) or of its faces along a."""
        e = [k == a for k in range(3)]
        K, J, I = torch.meshgrid(*[torch.arange(16 + e[k], device="cuda") for k in (2, 1, 0)], indexing="ij")
        return [(16 * self.where[:, k].clamp(min=0)[:, None] + t.reshape(1, -1)).reshape(-1) for k, t in enumerate((I, J, K))]

    def local(self, a):
        """The pool's faces along a: their coordinate along a in their block, 0 to 16."""
        return self.coords(a)[a] - 16 * self.where[:, a].clamp(min=0).repeat_interleave(sparse.BFACES)

    @staticmethod
    def place(c, shape):
        return (c[2] * shape[1] + c[1]) * shape[2] + c[0]

    def face_shape(self, a):
        return tuple(self.n[k] + (k == a) for k in (2, 1, 0))

    def faces(self, pattern):
        return [(_view(self.s, pattern % ax + "_F", self.nface).double(), _view(self.s, pattern % ax + "_C").double()) for ax in AX]

    def cells(self, name):
        return _view(self.s, name + "_F", self.ncell).double(), _view(self.s, name + "_C").double()

    def named(self, pattern, u):
        return {pattern % ax + p: t for ax, pair in zip(AX, u) for p, t in zip(("_F", "_C"), pair)}

    def named_cells(self, name, pair):
        return {name + p: t for p, t in zip(("_F", "_C"), pair)}

    def whole(self, a, u):
        """A face field's pool on the whole grid, the upper block's copy of a shared face, and
        where there is a face."""
        at, top, ok = self.place(self.coords(a), self.face_shape(a)), self.local(a) == 16, self.livemask(sparse.BFACES)
        g = torch.zeros(math.prod(self.face_shape(a)), dtype=F64, device="cuda")
        present = torch.zeros(g.shape, dtype=torch.bool, device="cuda")
        for part in (ok & top, ok & ~top):
            i = part.nonzero()[:, 0]
            g = g.index_copy(0, at[i], u[0][i])
            present[at[i]] = True
        return g, present

    def restrict_cells(self, fine, coarse):
        g = torch.zeros(math.prod(self.cell_shape), dtype=F64, device="cuda")
        ok = self.livemask(sparse.BCELLS)
        g[self.cell_at[ok]] = fine[ok]
        n = self.nc
        mean = g.view(n[2], 4, n[1], 4, n[0], 4).mean((1, 3, 5)).reshape(-1)
        return torch.where(self.covered, mean, coarse)

    def restrict_faces(self, a, u):
        """The coarse grid's faces with all 16 fine faces there take their mean."""
        g, present = self.whole(a, u)
        view = []
        for t in (g, present.double()):
            t = t.view(self.face_shape(a))
            t = t[tuple(slice(None, None, 4) if k == a else slice(None) for k in (2, 1, 0))]
            for k in range(3):
                if k != a:
                    d = 2 - k
                    t = t.unflatten(d, (self.nc[k], 4)).mean(d + 1)
            view.append(t.reshape(-1))
        return u[0], torch.where(view[1] > 0.999, view[0], u[1])

    def union(self, P, dt, phi0):
        phi = torch.minimum(phi0[0] + self.dx, _splat(self, P, dt)[self.cell_at])
        phi = torch.where(self.livemask(sparse.BCELLS), phi, _view(self.s, "PHI_F", self.ncell).double())
        return phi, self.restrict_cells(phi, phi0[1])

    def face_phi(self, a, phi):
        """The level set at the pool's faces: the mean of the two fine cells where the eight
        taps of its sample are fine, else the coarse grid's. Which taps those are is a matter
        of FP32 rounding (a face's centre lies on cell centres along two axes)."""
        c = self.coords(a)
        f32 = [torch.tensor(x, dtype=torch.float32, device="cuda") for x in self.lo]
        dx = torch.tensor(self.dx, dtype=torch.float32, device="cuda")
        pos = [f32[k] + (c[k].float() + _offset(k, a)) * dx for k in range(3)]
        tap = [torch.floor((pos[k] - f32[k]) / dx - 0.5).long() for k in range(3)]
        fine = torch.ones(c[0].shape, dtype=torch.bool, device="cuda")
        for m in range(8):
            t = [tap[k] + (m >> k & 1) for k in range(3)]
            for k in range(3):
                fine &= (t[k] >= 0) & (t[k] < self.n[k])
            fine &= self.pool[self.place([x.clamp(0, self.n[k] - 1) for k, x in enumerate(t)], self.cell_shape)] >= 0
        lo, hi = list(c), list(c)
        lo[a] = c[a] - 1
        both = [self.pool[self.place([x.clamp(0, self.n[k] - 1) for k, x in enumerate(t)], self.cell_shape)].long() for t in (lo, hi)]
        mean = 0.5 * (phi[0][both[0]] + phi[0][both[1]])
        i, w = [], []
        for k in range(3):
            q = ((pos[k] - f32[k]) / (4 * dx) - 0.5).double().clamp(0.0, self.nc[k] - 1.0)
            i.append(q.long().clamp(max=self.nc[k] - 2))
            w.append(q - i[k])
        coarse = 0.0
        shape = (self.nc[2], self.nc[1], self.nc[0])
        for m in range(8):
            at = self.place([i[k] + (m >> k & 1) for k in range(3)], shape)
            coarse = coarse + phi[1][at] * math.prod(w[k] if m >> k & 1 else 1.0 - w[k] for k in range(3))
        return torch.where(fine, mean, coarse)

    def blend(self, mom, wt, u0, phi):
        full, deep, out = float(self.s.nmin), (self.s.band - 1) * self.dx, []
        for a in range(3):
            at = self.place(self.coords(a), self.face_shape(a))
            m, w = mom[a][at], wt[a][at]
            mixed = (m + (full - w).clamp(min=0.0) * u0[a][0]) / w.clamp(min=full)
            ok = self.livemask(sparse.BFACES) & (self.face_phi(a, phi) >= -deep)
            out.append(self.restrict_faces(a, (torch.where(ok, mixed, u0[a][0]), u0[a][1])))
        return out


class _Conjugate(torch.autograd.Function):
    """A^-1 b by Jacobi-preconditioned CG, with its (symmetric) adjoint."""

    @staticmethod
    def forward(ctx, b, system, tol):
        ctx.system, ctx.tol = system, tol
        return system.cg(b, tol)

    @staticmethod
    def backward(ctx, g):
        return ctx.system.cg(g, ctx.tol), None, None


class _Faces:
    """Faces as the projection sees them: their places in u (axis, and 0 for the fine pool or
    the one grid, 1 for the coarse grid), the two cells, whether both are there, the distance
    between the cells and their coupling. `rows` says which of the cells' rows take the face
    from here and `sides` which cells' divergence does (a face between fine blocks is stored
    by both, and each copy serves its own block's cell)."""

    def __init__(self, a, which, lo, hi, inside, dist, coupling, rows, sides):
        self.a, self.which, self.lo, self.hi, self.inside = a, which, lo, hi, inside
        self.dist, self.coupling, self.rows, self.sides = dist, coupling, rows, sides


class _Poisson:
    """The projection's operator, assembled face by face; cells number the fine pool, then
    the coarse grid."""

    def __init__(self, G):
        self.G, self.groups, h = G, [], G.dx

        def full(n, x):
            return torch.full((n,), x, dtype=F64, device="cuda")

        if isinstance(G, _Dense):
            self.split, self.type, self.phi = None, _view(G.s, "TYPES").long(), G.cells("PHI")
            N = self.type.numel()
            dead = torch.zeros(N, dtype=torch.bool, device="cuda")
            self.scale, self.source = full(N, h), full(N, h * h)
            self.regular(G.n, 0, 0, ~dead, h, 1.0)
        else:
            nf, nc = G.ncell, math.prod(G.nc)
            self.split = nf
            self.type = torch.cat([_view(G.s, "TYPES_F", nf), _view(G.s, "TYPES_C")]).long()
            self.phi = torch.cat(G.cells("PHI"))
            dead = torch.cat([~G.livemask(sparse.BCELLS), G.covered])
            self.scale = torch.cat([full(nf, h), full(nc, 16 * h)])
            self.source = torch.cat([full(nf, h * h), full(nc, 64 * h * h)])
            self.blocks()
            self.regular(G.nc, 1, nf, ~G.covered, 4 * h, 4.0)
        self.liquid = (self.type == LIQUID) & ~dead
        self.diag = full(self.type.numel(), 0.0)
        rows, cols, vals = [], [], []
        for f in self.groups:
            for row, col, own in ((f.lo, f.hi, f.rows[0]), (f.hi, f.lo, f.rows[1])):
                i = (own & self.liquid[row] & (self.type[col] == LIQUID)).nonzero()[:, 0]
                rows.append(row[i])
                cols.append(col[i])
                vals.append(f.coupling[i])
                self.diag.index_add_(0, row[i], f.coupling[i])
                i = (own & self.liquid[row] & (self.type[col] == AIR)).nonzero()[:, 0]
                self.diag.index_add_(0, row[i], f.coupling[i] / _theta(self.phi[row[i]], self.phi[col[i]]))
        self.rows, self.cols, self.vals = torch.cat(rows), torch.cat(cols), torch.cat(vals)
        self.safe = torch.where(self.liquid & (self.diag > 0), self.diag, 1.0)

    def regular(self, n, which, first, there, dist, coupling):
        for a in range(3):
            lo, hi, has_lo, has_hi = _grid_faces(n, a)
            ok = has_lo & has_hi & there[lo] & there[hi]
            self.groups.append(_Faces(a, which, first + lo, first + hi, ok, torch.full(lo.shape, dist, dtype=F64, device="cuda"),
                                      torch.full(lo.shape, coupling, dtype=F64, device="cuda"), (ok, ok), (has_lo, has_hi)))

    def blocks(self):
        G, nf, h = self.G, self.G.ncell, self.G.dx
        for a in range(3):
            c, local, live = G.coords(a), G.local(a), G.livemask(sparse.BFACES)
            ends, inside = [], live.clone()
            for d in (1, 0):
                t = [c[k] - d * (k == a) for k in range(3)]
                inside &= (t[a] >= 0) & (t[a] < G.n[a])
                t = [x.clamp(0, G.n[k] - 1) for k, x in enumerate(t)]
                p = G.pool[G.place(t, G.cell_shape)].long()
                ends.append(torch.where(p >= 0, p, nf + G.place([x >> 2 for x in t], (G.nc[2], G.nc[1], G.nc[0]))))
            lo, hi = ends
            both = (lo < nf) & (hi < nf)
            own = (live & (local > 0), live & (local < 16))
            rows = (inside & (own[0] | (lo >= nf)), inside & (own[1] | (hi >= nf)))
            self.groups.append(_Faces(a, 0, lo, hi, inside, torch.where(both, h, 2.5 * h).double(),
                                      torch.where(both, 1.0, 0.4).double(), rows, own))

    def apply(self, x):
        return (self.diag * x).index_add_(0, self.rows, -self.vals * x[self.cols])

    def cg(self, b, tol):
        b = torch.where(self.liquid, b, 0.0)
        x, r = torch.zeros_like(b), b.clone()
        z = r / self.safe
        d, rho, stop = z.clone(), torch.dot(r, z), tol * torch.linalg.norm(b)
        for it in range(20000):
            if it % 20 == 0 and not torch.linalg.norm(r) > stop:
                break
            q = self.apply(d)
            alpha = rho / torch.dot(d, q)
            x += alpha * d
            r -= alpha * q
            z = r / self.safe
            new = torch.dot(r, z)
            d = z + (new / rho) * d
            rho = new
        return x

    def project(self, u, gamma, tol):
        """(u, P) after the projection; u per axis, a pair (fine, coarse) on the sparse basin."""
        parts = [list(t) if isinstance(t, tuple) else [t] for t in u]
        div = torch.zeros_like(self.scale)
        for f in self.groups:
            v = parts[f.a][f.which]
            for cell, own, sign in ((f.lo, f.sides[0], 1.0), (f.hi, f.sides[1], -1.0)):
                div = div.index_add(0, cell, torch.where(own, sign * v, 0.0))
        b = torch.where(self.liquid, -self.scale * div + gamma * self.source, 0.0)
        p = _Conjugate.apply(b, self, tol)
        for f in self.groups:
            tl, th, fl, fh = self.type[f.lo], self.type[f.hi], self.phi[f.lo], self.phi[f.hi]
            ok = f.inside & (tl != SOLID) & (th != SOLID) & ((tl == LIQUID) | (th == LIQUID))
            d = torch.where((tl == LIQUID) & (th == LIQUID), p[f.hi] - p[f.lo],
                            torch.where(tl == LIQUID, -p[f.lo] / _theta(fl, fh), p[f.hi] / _theta(fh, fl)))
            v = parts[f.a][f.which]
            parts[f.a][f.which] = torch.where(ok, v - d / f.dist, v)
        if self.split is None:
            return [t[0] for t in parts], p
        return [self.G.restrict_faces(a, tuple(t)) for a, t in enumerate(parts)], (p[:self.split], p[self.split:])


def _backward(G, P, pb, dt, tol):
    """The cotangents of the particles and of u0 behind G2P, the projection and P2G."""
    one = isinstance(G, _Dense)

    def leafs(u):
        return [t.detach().clone().requires_grad_() if one else tuple(x.detach().clone().requires_grad_() for x in t) for t in u]

    def flat(u):
        return list(u) if one else [x for t in u for x in t]

    def back(outs, seeds, ins):
        g = torch.autograd.grad(outs, ins, seeds, allow_unused=True)
        return [torch.zeros_like(i) if x is None else x for i, x in zip(ins, g)]

    def like(u, g):
        return g if one else [tuple(g[2 * a: 2 * a + 2]) for a in range(3)]

    # G2P at the particles: v where the grid was not reached passes through
    zero = [torch.zeros_like(t) if one else tuple(torch.zeros_like(x) for x in t) for t in G.faces("%s")]
    ok = _reached(G, P, G.faces("F%s"))
    ub = []
    for a in range(3):
        u = leafs(zero)
        whole, present = G.whole(a, u[a])
        val, row = _gather(G, P, a, whole, present)
        outs = [torch.where(ok, t, 0.0) for t in [val] + row]
        g = back(outs, [pb[VN[a]]] + [pb[CN[3 * a + k]] for k in range(3)], flat(u))
        ub.append(g[a] if one else tuple(g[2 * a: 2 * a + 2]))
    through = {f: torch.where(ok, 0.0, pb[f]) if f in VN else torch.zeros_like(pb[f]) for f in VN + CN}
    # the projection
    u = leafs(zero)
    un, _ = _Poisson(G).project(u, 0.0, 0.1 * tol)
    ub = like(u, back(flat(un), flat(ub), flat(u)))
    # P2G in v and the rows, and in u0, at the present level set
    Q = {f: (t.detach().clone().requires_grad_() if f in VN + CN else t) for f, t in P.items()}
    u0, phi = leafs(zero), G.cells("PHI")
    un = G.blend(*_deposit(G, Q, dt), u0, phi)
    g = back(flat(un), flat(ub), [Q[f] for f in VN + CN] + flat(u0))
    out = {"PB_" + f: through[f] + t for f, t in zip(VN + CN, g)}
    out.update(G.named("UB0_%s", like(u0, g[len(VN + CN):])))
    return out
