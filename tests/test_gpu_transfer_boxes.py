"""The tiled transfers' boxes on the dense basin: workgroups that are not full, particles
that take one box, several in turn, more than the kernels allow (left to the direct path),
and ones off the grid or not finite."""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu

VN = ("VX", "VY", "VZ")


def _particles(rng, g, n, places):
    """n particles in order round `places` clusters two cells wide."""
    lo, dx, dims = np.array(g.lo), g.dx, np.array(g.dims)
    at = rng.uniform(4, dims - 4, (places, 3))
    x = at[np.arange(n) * places // n] + rng.uniform(-1, 1, (n, 3))
    ps = {f: (lo[k] + x[:, k] * dx).astype(np.float32) for k, f in enumerate(("PX", "PY", "PZ"))}
    for f in VN + tuple("C%d" % k for k in range(9)):
        ps[f] = rng.normal(0, 0.5, n).astype(np.float32)
    ps["LAG"] = rng.uniform(-0.02, 0.02, n).astype(np.float32)
    return ps


# 1 and 7 clusters: one box and up to four in the deposit; 200: left to the direct path. 1000
# particles are four workgroups, the last with 232. 140,000 are 547, where the gather takes up
# to two boxes: two clusters a workgroup, three or four, and five or six (left to the direct path).
@pytest.mark.parametrize("n,places,off", [(1, 1, 0), (255, 1, 0), (257, 7, 1), (1000, 7, 0), (1000, 200, 3), (140000, 1094, 1),
                                          (140000, 1800, 0), (140000, 2700, 3)])
def test_boxes(mael, orc, ctx, n, places, off):
    print("case: boxes n=%d places=%d" % (n, places), flush=True)
    b = mael.Basin(radius=18.0, depth=12.0, Γ=225.0, core=2.5)
    s = mael.FlipBasin(b, dx=0.6, capacity=n + 1000)
    g, phi, u, v, w, _ = orc.dense_scene(18.0, 12.0, 3.0, 0.6, 225.0, 2.5)
    rng = np.random.default_rng(n + places)
    ps = _particles(rng, g, n, places)
    if off:   # one off the grid on either side; where there are more, far off it and not finite
        ps["PX"][n // 2] = np.float32(g.lo[0] - 30.0)
        if off > 1:
            ps["PY"][n // 3], ps["PZ"][n // 5] = np.float32(1e9), np.float32(np.inf)
    s.set_particles(ps, n)
    flags = []
    for name, arr in (("U", u), ("V", v), ("W", w)):
        s.set(name, arr)
        s.set(name + "0", arr)
        f = (rng.random(arr.shape) > 0.002).astype(np.uint8)
        s.set("F" + name, f)
        flags.append(f)
    s.set("PHI0", phi)
    dt = 0.04
    mael.particles2grid(s, dt)
    # the reference deposit of the particles that reach the grid (the others reach no node)
    keep = np.isfinite(ps["PZ"]) & (np.abs(ps["PY"]) < 1e8)
    sub = {f: a[keep] for f, a in ps.items()}
    rphi, _, _, _, M, Wt = orc.dense_p2g(g, sub, int(keep.sum()), dt, phi, u, v, w)
    assert np.array_equal(s.get("PHI").view(np.uint32), rphi.view(np.uint32))
    for a, ax in enumerate("UVW"):
        # a contribution is rounded to 2^-32 from FP32 products (five roundings of 2^-24 each)
        for got, ref in ((s.get("MOM_" + ax), M[a]), (s.get("WT_" + ax), Wt[a])):
            np.testing.assert_allclose(got * 2.0 ** -32, ref, rtol=0, atol=5 * 2.0 ** -24 * max(1.0, np.abs(ref).max()))
    for name, arr in (("U", u), ("V", v), ("W", w)):   # the gather reads the faces above, not the blend
        s.set(name, arr)
    mael.grid2particles(s, dt)
    ref = orc.dense_g2p(g, sub, int(keep.sum()), u, v, w, *flags, dt, 9.81)
    for f in VN + tuple("C%d" % k for k in range(9)):
        assert np.array_equal(s.get(f)[keep].view(np.uint32), ref[f].view(np.uint32)), f


# A particle's part of the adjoints does not depend on its workgroup's other particles: in
# shuffled order (up to 200 clusters a workgroup, most left to the direct path) it has the
# same bits as in the clusters' order, and so has the cotangent of the faces (whole numbers).
@pytest.mark.parametrize("n,places,off", [(1, 1, 0), (257, 7, 1), (1000, 7, 0), (1000, 200, 3), (140000, 1800, 3)])
def test_adjoint_boxes(mael, orc, ctx, n, places, off):
    print("case: adjoint boxes n=%d places=%d" % (n, places), flush=True)
    b = mael.Basin(radius=18.0, depth=12.0, Γ=225.0, core=2.5)
    s = mael.FlipBasin(b, dx=0.6, capacity=n + 1000)
    g = orc.dense_scene(18.0, 12.0, 3.0, 0.6, 225.0, 2.5)[0]
    rng = np.random.default_rng(n + places)
    ps = _particles(rng, g, n, places)
    if off:
        ps["PX"][n // 2] = np.float32(g.lo[0] - 30.0)
        if off > 1:
            ps["PY"][n // 3], ps["PZ"][n // 5] = np.float32(1e9), np.float32(np.inf)
    names = VN + tuple("C%d" % k for k in range(9))
    pbar = {f: rng.normal(0, 1, n).astype(np.float32) for f in names}
    flags = {"F" + c: (rng.random(s.shape(c)) > 0.002).astype(np.uint8) for c in "UVW"}
    ubar = {"UB_" + c: rng.normal(0, 1, s.shape(c)).astype(np.float32) for c in "UVW"}
    dt, got = 0.04, []
    for order in (np.arange(n), rng.permutation(n)):
        s.set_particles({f: a[order] for f, a in ps.items()}, n)
        for f, a in flags.items():
            s.set(f, a)
        for f, a in pbar.items():
            s.set("PB_" + f, a[order])
        mael.grid2particles_adjoint(s, dt)
        back = np.argsort(order)
        out = [s.get("PB_" + f)[back] for f in names] + [s.get("UB_" + c) for c in "UVW"]
        s.set("PHI", np.zeros(s.shape("PHI"), np.float32))   # every face in the band
        for f, a in ubar.items():
            s.set(f, a)
        for f in names:
            s.set("PB_" + f, np.zeros(n, np.float32))
        mael.particles2grid_adjoint(s, dt)
        got.append(out + [s.get("PB_" + f)[back] for f in names])
    assert any(a.any() for a in got[0][-12:])
    for a, b in zip(*got):
        assert np.array_equal(a.view(np.uint32), b.view(np.uint32))
