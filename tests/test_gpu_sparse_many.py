"""More than 1,024 live fine blocks, where the per-slot kernels take a workgroup a slot instead
of several (and the transfers' launches one workgroup for the three components): the same
checks against the CPU oracle as on the 60 cm scenes, on a 20 cm basin with all of its 1,152
blocks refined. The extrapolation, which the oracle does not have, gives a block the same bits
whether the basin holds many slots or few."""
import numpy as np
import pytest

from test_gpu_sparse import BCELLS, BFACES, _basin, _check_projected, _fine, _projection_inputs, _scene, _upload

pytestmark = pytest.mark.gpu


@pytest.fixture(scope="module")
def M():
    import maelstrom_amd
    return maelstrom_amd


@pytest.fixture(scope="module")
def scene():
    """The oracle's scene; each test uploads the state it finds."""
    o = _scene(dx=0.2, blocks=1200, capacity=1_500_000)
    o.refine(np.ones(int(np.prod(list(o.grid.nb))), np.uint8))
    assert o.nslots == 1152
    o.classify()
    return o


def test_p2g(M, scene):
    """883,000 particles: a workgroup takes the three components (above 512 workgroups)."""
    o = scene
    assert o.n > 512 * 256
    print("case: sparse p2g, %d slots, %d particles" % (o.nslots, o.n), flush=True)
    rng = np.random.default_rng(3)
    for nm in ["vx", "vy", "vz"] + ["c%d" % k for k in range(9)]:
        o.array(nm)[:o.n] += rng.normal(0, 0.3, o.n).astype(np.float32)
    s = _upload(M, o)
    dt = np.float32(0.05)
    M.sparse.particles2grid(s, dt)
    momwt = o.p2g(dt, momwt=True)
    F = o.nslots * BFACES
    for a, nm in enumerate("UVW"):   # bars as test_p2g_parity's: FP32 products rounded to 2^-32
        for got, ref in ((s.get("MOM_" + nm), momwt[a][:F]), (s.get("WT_" + nm), momwt[3 + a][:F])):
            np.testing.assert_allclose(got * 2.0 ** -32, ref, rtol=0, atol=1e-6 * max(1.0, np.abs(ref).max()))
    np.testing.assert_array_equal(s.get("PHI_F"), _fine(o, "phi_f", BCELLS))
    for nm in "uvw":
        exp = _fine(o, nm + "_f", BFACES)
        assert np.linalg.norm(s.get(nm.upper() + "_F") - exp) <= 1e-6 * np.linalg.norm(exp), nm


def test_redistance(M, scene):
    o = scene
    print("case: sparse redistance, %d slots" % o.nslots, flush=True)
    s = _upload(M, o)
    M.sparse.redistance(s, 3)
    o.redistance(3)
    np.testing.assert_array_equal(s.get("PHI_F").view(np.uint32), _fine(o, "phi_f", BCELLS).view(np.uint32))
    np.testing.assert_array_equal(s.get("PHI_C").ravel().view(np.uint32), o.array("phi_c").view(np.uint32))


@pytest.mark.parametrize("many", [False, True])
def test_walls(M, scene, many):
    """Without layers, and every face reached, `extrapolate!` closes the walls' faces alone."""
    from maelstrom_amd import _lib as L
    o = scene if many else _scene()
    print("case: sparse walls, %d slots" % o.nslots, flush=True)
    rng = np.random.default_rng(4)
    for nm in ("u_f", "v_f", "w_f"):
        arr = o.array(nm)
        arr[:] += rng.normal(0, 0.3, arr.size).astype(np.float32)
    o.fill_flags(1)
    s = _upload(M, o)
    s.ctx.check(L.lib().mael_sparse_extrapolate(s.h, 0, 0, 0))
    before = _fine(o, "u_f", BFACES).copy()
    o.solidify()
    assert (before != _fine(o, "u_f", BFACES)).any()
    for nm in "uvw":
        np.testing.assert_array_equal(s.get(nm.upper() + "_F").view(np.uint32), _fine(o, nm + "_f", BFACES).view(np.uint32))


def test_project(M, scene):
    """The couplings and the faces' pressure differences, from the FP32 and the FP64 pressure.
    The solves start from the oracle's pressure rounded to FP32, and the flexible CG does not
    raise the error's energy norm, so the bar is not the residual's through this larger
    system's condition."""
    o = scene
    print("case: sparse project, %d slots" % o.nslots, flush=True)
    o.classify()
    _projection_inputs(o)
    tried = [(refine, _upload(M, o)) for refine in (0, 10)]
    o.project(gamma=0.01, tol=1e-10, maxiter=600, policy=0)
    for refine, s in tried:
        s.set("P_F", _fine(o, "P_f", BCELLS))
        s.set("P_C", o.array("P_c"))
        st = M.sparse.project(s, 0.1, gamma=0.01, tol=1e-6, maxiter=400, policy=0, boost=1.0, refine=refine)
        assert st.rel_residual <= 1.01e-6, (refine, st.rel_residual)
        _check_projected(o, s)


def _basin_of(M, blocks, rng):
    """A 20 cm basin with those blocks live, their slots in random order."""
    s = M.SparseBasin(_basin(M), dx=0.2, blocks=1200, capacity=200_000)
    nb = tuple(int(x) for x in s.grid.nb)
    slot, where = np.zeros(s.nblocks, np.int32), np.full((1200, 3), -1, np.int32)
    for k, b in enumerate(rng.permutation(blocks)):
        slot[b] = k + 1
        where[k] = (b % nb[0], (b // nb[0]) % nb[1], b // (nb[0] * nb[1]))
    s.set_topology(slot, where, len(blocks))
    return s, slot[blocks] - 1


@pytest.mark.parametrize("layers,kick", [(6, 1), (5, 0), (1, 1)])
def test_extrapolate_many_and_few(M, layers, kick):
    """A plane of blocks left out parts the basin: the blocks on either side take the values
    that they take in a basin of that side alone (480 and 576 live slots: three axes and 17
    workgroups a slot a launch)."""
    from maelstrom_amd import _lib as L
    print("case: sparse extrapolate, layers %d kick %d" % (layers, kick), flush=True)
    rng = np.random.default_rng(layers)
    N = 12 * 12 * 8
    bx = np.arange(N) % 12
    value = {ax: rng.normal(0, 1, (N, BFACES)).astype(np.float32) for ax in "UVW"}
    older = {ax: rng.normal(0, 1, (N, BFACES)).astype(np.float32) for ax in "UVW"}
    flag = {ax: (rng.random((N, BFACES)) < (0.02 if layers > 1 else 0.5)).astype(np.uint8) for ax in "UVW"}
    # particles in the third and the ninth layer of blocks along x, clear of the part left out
    n = 20_000
    unit = rng.random((n, 3))

    def run(keep):
        blocks = np.flatnonzero(keep)
        s, at = _basin_of(M, blocks, rng)
        lo, dx = np.array(s.grid.lo), 0.2

        def put(name, per_block):
            a = np.zeros((len(blocks), BFACES), per_block.dtype)
            a[at] = per_block[blocks]
            s.set(name, a)
        for ax in "UVW":
            put(ax + "_F", older[ax])
            s.set(ax + "_C", np.zeros(s.shape(ax + "_C"), np.float32))
        s.ctx.check(L.lib().mael_sparse_save_reflect(s.h))
        for ax in "UVW":
            put(ax + "_F", value[ax])
            put("F" + ax + "_F", flag[ax])
        s.ctx.check(L.lib().mael_sparse_extrapolate(s.h, layers, 2, kick))
        out = {f: s.get(f).reshape(-1, BFACES)[at] for ax in "UVW" for f in (ax + "_F", "F" + ax + "_F")}
        if kick:   # the reflected flow, which the gather reads
            x = unit * [16, 12 * 16, 8 * 16]
            x[:, 0] += np.where(np.arange(n) % 2, 2 * 16, 9 * 16)
            ps = {"PX": lo[0] + x[:, 0] * dx, "PY": lo[1] + x[:, 1] * dx, "PZ": lo[2] + x[:, 2] * dx}
            for f in ["VX", "VY", "VZ", "LAG"] + ["C%d" % k for k in range(9)]:
                ps[f] = np.zeros(n)
            s.set_particles(ps, n)
            s.ctx.check(L.lib().mael_sparse_set_flow(s.h, 1))
            M.sparse.grid2particles(s, 0.05)
            out["v"] = s.get("VX")
        return blocks, out

    blocks, got = run(bx != 5)
    assert len(blocks) == 1056
    changed = 0
    for side in (bx < 5, bx > 5):
        few, ref = run(side)
        where = np.searchsorted(blocks, few)
        for f in ref:
            if f == "v":
                mine = np.arange(n) % 2 == (1 if side[0] else 0)
                assert np.unique(ref[f][mine]).size > n // 10
                np.testing.assert_array_equal(got[f][mine].view(np.uint32), ref[f][mine].view(np.uint32))
            else:
                np.testing.assert_array_equal(got[f][where].view(np.uint8), ref[f].view(np.uint8), err_msg=f)
                changed += int(f[0] == "F" and (ref[f] != flag[f[1]][few]).any())
    assert changed == 6   # layers were made
