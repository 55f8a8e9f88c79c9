"""The V-cycles' small levels, which share launches.

The dense levels of the sparse basin's V-cycle on grids whose levels take each of their
launches: tiles of 8^3 and 16x8x8 cells with remainders, a launch a sweep (the largest
level, and more than one pair of sweeps), the one-workgroup tail of one, two and three
levels, and an odd coarsest level. No fine blocks: the composite levels are the coarse grid."""
import ctypes as C

import numpy as np
import pytest

import oracle as O

pytestmark = pytest.mark.gpu

# radius, depth -> the coarse grid; V-cycle levels follow by halves to at most 1024 cells
CASES = {
    "one level, 16^3 halved once": (18.0, 12.0, (16, 16, 16)),
    "8^3 tiles and an odd coarsest level, 112x112x48 .. 14x14x6, 7x7x3": (125.0, 85.0, (112, 112, 48)),
    "16x8x8 tiles, 80x80x32 .. 10x10x4": (90.0, 60.0, (80, 80, 32)),
}


@pytest.mark.parametrize("precision,sweeps", [(0, 1), (0, 2), (1, 1), (2, 1)])
@pytest.mark.parametrize("case", sorted(CASES))
def test_levels_match_oracle(mael, case, precision, sweeps):
    radius, depth, dims = CASES[case]
    print("case: %s precision %d sweeps %d" % (case, precision, sweeps), flush=True)
    o = O.SparseOracle(radius, depth, 3.0, 0.6, 2, 1, 16, 4, 8)
    g = o.grid
    rmax = np.float32(np.hypot(np.float32(g.lo[0]), np.float32(g.lo[1])))
    o.init_coarse(O.surface_table(225.0, 2.5, 9.81, rmax), rmax, 225.0, 2.5)
    o.classify()
    s = mael.SparseBasin(mael.Basin(radius=radius, depth=depth, Γ=225.0, core=2.5), dx=0.6, blocks=1, capacity=16)
    assert s.nc == dims
    s.set("PHI_C", o.array("phi_c"))
    s.set("TYPES_C", o.array("types_c"))
    rng = np.random.default_rng(5)
    rc = np.where(o.array("types_c") == 1, rng.normal(0, 1, o.array("types_c").size), 0).astype(np.float32)
    s.set("RHS_C", rc)
    opts = mael.sparse.solve_options(precision=precision, boost=1.0, sweeps=sweeps)
    s.ctx.check(mael.lib().mael_sparse_vcycle(s.h, C.byref(opts), 0))
    z = s.get("P_C").ravel().astype(np.float64)
    _, ze = o.vcycle(np.zeros(o.array("P_f").size, np.float32), rc, sweeps=sweeps, coarse=opts.coarse, boost=1.0)
    err = np.linalg.norm(z - ze) / np.linalg.norm(ze)
    print("rel L2 vs FP64 oracle %.3e" % err, flush=True)
    # the storage's rounding (2^-24, 2^-11, 2^-8) through a few tens of passes
    assert err < {0: 1e-5, 1: 3e-3, 2: 2e-2}[precision], err


def test_levels_subnormal(mael):
    """A right-hand side of 2^-140 and below: the coarsest solve meets subnormal quotients and is
    made again with divisions. Its values are some hundreds of the smallest number, to half of
    one in each of a few tens of passes."""
    radius, depth, dims = CASES["one level, 16^3 halved once"]
    print("case: subnormal right-hand side", flush=True)
    o = O.SparseOracle(radius, depth, 3.0, 0.6, 2, 1, 16, 4, 8)
    g = o.grid
    rmax = np.float32(np.hypot(np.float32(g.lo[0]), np.float32(g.lo[1])))
    o.init_coarse(O.surface_table(225.0, 2.5, 9.81, rmax), rmax, 225.0, 2.5)
    o.classify()
    s = mael.SparseBasin(mael.Basin(radius=radius, depth=depth, Γ=225.0, core=2.5), dx=0.6, blocks=1, capacity=16)
    assert s.nc == dims
    s.set("PHI_C", o.array("phi_c"))
    s.set("TYPES_C", o.array("types_c"))
    rng = np.random.default_rng(8)
    rc = np.where(o.array("types_c") == 1, rng.uniform(0, 2.0 ** -140, o.array("types_c").size), 0).astype(np.float32)
    s.set("RHS_C", rc)
    opts = mael.sparse.solve_options(precision=0, boost=1.0, sweeps=1)
    s.ctx.check(mael.lib().mael_sparse_vcycle(s.h, C.byref(opts), 0))
    z = s.get("P_C").ravel().astype(np.float64)
    _, ze = o.vcycle(np.zeros(o.array("P_f").size, np.float32), rc, sweeps=1, coarse=opts.coarse, boost=1.0)
    err = np.linalg.norm(z - ze) / np.linalg.norm(ze)
    print("rel L2 vs FP64 oracle %.3e, largest %.3g units" % (err, np.abs(ze).max() * 2.0 ** 149), flush=True)
    assert err < 2e-2, err


# radius, depth, top, dx -> cells; the dense V-cycle's levels halve them to at most 1024
DENSE = {
    "tiles and a 2,048-cell tail, 64x64x32 .. 8x8x4": (18.0, 12.0, 3.0, 0.6, (64, 64, 32)),
    "tile remainders and a 4,840-cell tail, 44x44x20 .. 11x11x5": (4.0, 2.0, 1.5, 0.2, (44, 44, 20)),
    "a level too wide for the tail, 128x128x4 .. 32x32x1": (36.9, 0.6, 0.9, 0.6, (128, 128, 4)),
    "tiles off by half, 40x40x24 .. 10x10x6": (10.2, 8.0, 5.0, 0.6, (40, 40, 24)),
    "two levels, the tail the whole V-cycle, 18x18x8 .. 9x9x4": (4.0, 2.0, 1.5, 0.6, (18, 18, 8)),
    "one level, the coarsest solve alone, 9x8x7": (4.0, 2.0, 1.5, 0.6, (9, 8, 7)),
}


@pytest.mark.parametrize("sweeps,queued", [(1, 0), (2, 0), (2, 1), (3, 1)])
@pytest.mark.parametrize("case", sorted(DENSE))
def test_dense_levels_bits(mael, orc, monkeypatch, case, sweeps, queued):
    """The dense basin's V-cycle on random cell types (empty rows and single-cell pools among
    them) in the oracle's FP32 V-cycle's bits: both take every sum and division in the
    reference's order."""
    radius, depth, top, dx, dims = DENSE[case]
    print("case: %s sweeps %d queued %d" % (case, sweeps, queued), flush=True)
    g = orc.flipgrid(radius, depth, top, dx)
    if case.startswith("one level"):   # flipgrid makes two or more; the C ABI takes one
        g.n[:], g.levels = dims, 1
        one = mael.flipgrid(mael.Basin(radius=radius, depth=depth, rimwall=top), dx)
        one.n[:], one.levels = dims, 1
        monkeypatch.setattr(mael.dense, "flipgrid", lambda *a: one)
    assert g.dims == dims
    s = mael.FlipBasin(mael.Basin(radius=radius, depth=depth, rimwall=top), dx=dx, capacity=16)
    rng = np.random.default_rng(3)
    shape = orc.cells_shape(g)
    types = rng.choice(np.array([0, 1, 2], np.uint8), shape, p=[0.25, 0.65, 0.1])
    phi = (rng.uniform(0.01, 1.0, shape) * np.where(types == 1, -1, 1)).astype(np.float32)
    r = np.where(types == 1, rng.normal(0, 1, shape), 0).astype(np.float32)
    for name, a in (("TYPES", types), ("PHI", phi), ("RHS", r)):
        s.set(name, a)
    opts = mael.dense.solve_options(sweeps=sweeps)
    s.ctx.check(mael.lib().mael_dense_vcycle(s.h, C.byref(opts), queued))
    z = s.get("P")
    ref = orc.dense_vcycle(g, types, phi, r, sweeps=sweeps, fp32=True)
    assert np.array_equal(z.view(np.uint32), ref.view(np.uint32)), int((z.view(np.uint32) != ref.view(np.uint32)).sum())
