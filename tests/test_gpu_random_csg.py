"""Seeded random CSG shapes against the oracle (NormalMultiPlaneShape,
NormalCylindricalShape, NormalIntersectionShape and NormalUnionShape of
NM/JMONSEL): rotated boxes and finite cylinders, 2 to 8 of them, joined by
random unions and intersections, as one PMMA region in the chamber.  The
device's convex primitives + truth-table walk against the oracle's
depth-counter walk of the reference's shapes: the region containing a point
(RegionBase::containingSubRegion) and findEndOfStep (RegionBase.cu:74-119)
on 20,000 random segments per shape, up to half of them from inside it; and
electron transport through three of them (yields within 3 sigma, exit
histograms by KS), which also runs the safety bound that lets steps skip
findEndOfStep on shapes it was not built around.  Nested scenes put a
random Si region inside a random PMMA one, with a random PMMA sibling beside
them, so that locating descends a region tree and findEndOfStep tests a
region's own shape and its children's."""
import numpy as np
import pytest

import stats_util as su

pytestmark = pytest.mark.gpu

NM = 1e-9


def _rotation(rng):
    q = rng.normal(size=4)
    w, x, y, z = q / np.linalg.norm(q)
    return np.array([[1 - 2 * (y * y + z * z), 2 * (x * y - z * w), 2 * (x * z + y * w)],
                     [2 * (x * y + z * w), 1 - 2 * (x * x + z * z), 2 * (y * z - x * w)],
                     [2 * (x * z - y * w), 2 * (y * z + x * w), 1 - 2 * (x * x + y * y)]])


def random_shape(M, rng, n_leaves, hold):
    """A random CSG tree of n_leaves convex parts within about 35 nm of the
    origin; every object goes to `hold` (the host classes keep pointers)."""
    def leaf():
        c = rng.uniform(-8.0, 8.0, 3)
        if rng.random() < 0.5:
            R = _rotation(rng)
            h = rng.uniform(6.0, 20.0, 3)
            s = M.NormalMultiPlaneShape()
            for i in range(3):
                for sgn in (1.0, -1.0):
                    n = sgn * R[:, i]
                    s.addPlane(list(n), list((c + n * h[i]) * NM))
        else:
            a = rng.normal(size=3)
            a /= np.linalg.norm(a)
            half = rng.uniform(6.0, 20.0)
            s = M.NormalCylindricalShape(list((c - a * half) * NM), list((c + a * half) * NM),
                                         float(rng.uniform(3.0, 12.0)) * NM)
        hold.append(s)
        return s

    def build(n):
        if n == 1:
            return leaf()
        k = int(rng.integers(1, n))
        a, b = build(k), build(n - k)
        s = M.NormalUnionShape(a, b) if rng.random() < 0.5 else M.NormalIntersectionShape(a, b)
        hold.append(s)
        return s

    return build(n_leaves)


def nested_csg_scene(M, seed):
    """chamber -> A (PMMA, 3 parts) -> B (Si, 2 parts); chamber -> C (PMMA,
    2 parts, 25 nm along x)."""
    from cudamonsel_amd import scenes
    rng = np.random.default_rng(seed)
    sc = scenes.Scene()
    ch = scenes._chamber(sc)
    hold = []
    a = random_shape(M, rng, 3, hold)
    b = random_shape(M, rng, 2, hold)
    c = random_shape(M, rng, 2, hold)
    M.NShapes.translate(c, [25.0 * NM, 0.0, 0.0])
    ra = M.Region(ch, scenes.MATERIALS["PMMA"](sc), a)
    rb = M.Region(ra, scenes.MATERIALS["Si"](sc), b)
    rc = M.Region(ch, scenes.MATERIALS["PMMA"](sc), c)
    sc.hold(*hold, ra, rb, rc)
    scenes._finish(sc, 500.0, 0.5, 40.0)
    return sc


def csg_scene(M, seed, n_leaves, compat=True):
    from cudamonsel_amd import scenes
    rng = np.random.default_rng(seed)
    sc = scenes.Scene()
    ch = scenes._chamber(sc)
    msm = scenes.MATERIALS["PMMA"](sc)
    hold = []
    shape = random_shape(M, rng, n_leaves, hold)
    reg = M.Region(ch, msm, shape)
    sc.hold(*hold, reg)
    scenes._finish(sc, 500.0, 0.5, 40.0)   # the beam starts at z = -60 nm
    sc.monte.setRefCompat(M.MONSEL_COMPAT_REFERENCE if compat else M.MONSEL_COMPAT_FIXED)
    return sc


@pytest.mark.parametrize("seed", range(8))
def test_random_csg_geometry_against_oracle(oracle, M, seed):
    """Shape `seed` has 2 + seed convex parts (2 to 8 at seed 0 to 6, and 5
    again at seed 7 in fixed mode)."""
    from cudamonsel_amd.abi import probe_for
    n_leaves = 2 + seed if seed < 7 else 5
    sc = csg_scene(M, 1000 + seed, n_leaves, compat=seed < 7)
    pr, cs = probe_for(sc)
    osc = oracle.OracleScene(cs)
    rng = np.random.default_rng(seed)
    # segments start inside the shape for up to half of them (points drawn in
    # a 60 nm cube and sorted by the oracle), outside for the rest
    cand = rng.uniform(-30.0, 30.0, (400000, 3))
    where = osc.locate(cand)
    ins, outs = cand[where == 1], cand[where == 0]
    assert ins.shape[0] >= 300, ins.shape[0]           # the shape has volume
    n_in = min(10000, ins.shape[0])
    p0 = np.concatenate([ins[:n_in], outs[:20000 - n_in]])
    n = p0.shape[0]
    d = rng.normal(size=(n, 3))
    d /= np.linalg.norm(d, axis=1)[:, None]
    L = rng.uniform(0.5, 50.0, n)
    p1 = p0 + d * L[:, None]
    p0 = p0.astype(np.float32).astype(np.float64)
    p1 = p1.astype(np.float32).astype(np.float64)
    reg = osc.locate(p0)
    assert np.mean(pr.locate(p0) == reg) > 0.999
    agree = tot = crossings = 0
    for r in np.unique(reg):
        if r < 0:
            continue
        m = reg == r
        ou, onx, _ = osc.find_end_of_step(r, p0[m], p1[m])
        gu, gnx, _ = pr.find_end_of_step(r, p0[m], p1[m])
        hit = ou <= 1.0
        # crossing distance apart, for segments that cross (u is infinite otherwise)
        apart = np.zeros(hit.shape)
        apart[hit] = np.abs(ou[hit] - gu[hit].astype(np.float64)) * L[m][hit]
        ok = (onx == gnx) & (~hit | (apart < 1e-3))
        agree += ok.sum()
        tot += m.sum()
        crossings += hit.sum()
    # measured: 20,000 of 20,000 on seven shapes, 19,999 on one; the
    # allowance is for FP32 rounding of grazing crossings
    print(f"shape {seed}: findEndOfStep agreement {agree}/{tot}, {crossings} crossings")
    assert crossings > 300
    assert tot - agree <= 20, (agree, tot)


@pytest.mark.parametrize("seed,n_leaves", [(2001, 3), (2002, 5), (2003, 8)])
def test_random_csg_transport_against_oracle(oracle, M, seed, n_leaves):
    sc = csg_scene(M, seed, n_leaves)
    centers = np.array([[x * NM, y * NM, sc.beam_z] for x in np.linspace(-12.0, 12.0, 4)
                        for y in np.linspace(-12.0, 12.0, 4)])
    sc.monte.setSeed(seed)
    r = sc.monte.runPixels(centers, 500, 50, 50.0)
    o = oracle.OracleScene(sc.monte.compileScene()).run(centers, 500, M.ToSI.eV(500.0), 0.5e-9, seed=seed,
                                                        nbins=50, se_cutoff_eV=50.0, threads=0)
    assert r.stats.queue_overflow == 0 and r.stats.watchdog_drops == 0 and o["stats"]["watchdog_drops"] == 0
    zs, zb = su.total_z(su.from_gpu(r), su.from_oracle(o))
    assert abs(zs) < 3 and abs(zb) < 3, (zs, zb)
    for name in ("backEnergyHist", "elevationHist", "azimuthHist"):
        D, p = su.ks_binned(getattr(r, name), o[name])
        assert p > 0.01 / 3, (name, D, p)


@pytest.mark.parametrize("seed", [3001, 3002, 3003])
def test_nested_csg_geometry_and_transport_against_oracle(oracle, M, seed):
    from cudamonsel_amd.abi import probe_for
    sc = nested_csg_scene(M, seed)
    pr, cs = probe_for(sc)
    osc = oracle.OracleScene(cs)
    rng = np.random.default_rng(seed)
    cand = rng.uniform(-30.0, 50.0, (400000, 3)) * np.array([1.0, 0.75, 0.75])
    where = osc.locate(cand)
    regions = [r for r in np.unique(where) if r > 0]
    assert len(regions) == 3, regions                  # every region has volume
    parts = [cand[where == r][:4000] for r in regions]
    p0 = np.concatenate(parts + [cand[where == 0][:20000 - sum(x.shape[0] for x in parts)]])
    n = p0.shape[0]
    d = rng.normal(size=(n, 3))
    d /= np.linalg.norm(d, axis=1)[:, None]
    L = rng.uniform(0.5, 50.0, n)
    p1 = p0 + d * L[:, None]
    p0 = p0.astype(np.float32).astype(np.float64)
    p1 = p1.astype(np.float32).astype(np.float64)
    reg = osc.locate(p0)
    assert np.sum(pr.locate(p0) != reg) <= 20
    agree = tot = 0
    for r in np.unique(reg):
        if r < 0:
            continue
        m = reg == r
        ou, onx, _ = osc.find_end_of_step(r, p0[m], p1[m])
        gu, gnx, _ = pr.find_end_of_step(r, p0[m], p1[m])
        hit = ou <= 1.0
        apart = np.zeros(hit.shape)
        apart[hit] = np.abs(ou[hit] - gu[hit].astype(np.float64)) * L[m][hit]
        agree += ((onx == gnx) & (~hit | (apart < 1e-3))).sum()
        tot += m.sum()
    print(f"nested {seed}: findEndOfStep agreement {agree}/{tot}")
    assert tot - agree <= 20, (agree, tot)
    centers = np.array([[x * NM, 0.0, sc.beam_z] for x in np.linspace(-10.0, 35.0, 16)])
    sc.monte.setSeed(seed)
    g = sc.monte.runPixels(centers, 500, 50, 50.0)
    o = osc.run(centers, 500, M.ToSI.eV(500.0), 0.5e-9, seed=seed, nbins=50, se_cutoff_eV=50.0, threads=0)
    assert g.stats.queue_overflow == 0 and g.stats.watchdog_drops == 0 and o["stats"]["watchdog_drops"] == 0
    zs, zb = su.total_z(su.from_gpu(g), su.from_oracle(o))
    assert abs(zs) < 3 and abs(zb) < 3, (zs, zb)


@pytest.mark.parametrize("n", [2, 3, 5, 8])
def test_walk_through_a_row_of_overlapping_boxes(oracle, M, n):
    """The union of n boxes 12 nm long, each overlapping the next by 2 nm, is
    one box: a segment along it passes up to 2 n - 2 crossings inside the
    shape, each a pass of the walk over the parts that are left on the
    segment.  Against the oracle's findEndOfStep of that one box; segments in
    every direction, a third of them along the row and some of those from
    outside.  (FP32 distances of some tens of nm: 1e-3 nm; the faces' normals
    are axis vectors, exact in FP32.)"""
    from cudamonsel_amd import scenes
    from cudamonsel_amd.abi import probe_for

    def box(hold, x0, x1):
        s = M.NormalMultiPlaneShape()
        for nrm, p in (([1, 0, 0], [x1, 0, 0]), ([-1, 0, 0], [x0, 0, 0]), ([0, 1, 0], [0, 9, 0]),
                       ([0, -1, 0], [0, -9, 0]), ([0, 0, 1], [0, 0, 7]), ([0, 0, -1], [0, 0, -7])):
            s.addPlane([float(v) for v in nrm], [v * NM for v in p])
        hold.append(s)
        return s

    def scene(parts):
        sc = scenes.Scene()
        ch = scenes._chamber(sc)
        hold = []
        shape = box(hold, *parts[0])
        for p in parts[1:]:
            shape = M.NormalUnionShape(shape, box(hold, *p))
            hold.append(shape)
        reg = M.Region(ch, scenes.MATERIALS["PMMA"](sc), shape)
        sc.hold(*hold, reg)
        scenes._finish(sc, 500.0, 0.5, 40.0)
        sc.monte.setRefCompat(M.MONSEL_COMPAT_FIXED)
        return sc

    row = scene([(10.0 * k, 10.0 * k + 12.0) for k in range(n)])
    pr, _ = probe_for(row)
    whole = scene([(0.0, 10.0 * n + 2.0)])
    osc = oracle.OracleScene(whole.monte.compileScene())
    rng = np.random.default_rng(n)
    m = 6000
    L = rng.uniform(1.0, 12.0 * n, m)
    d = rng.normal(size=(m, 3))
    d[::3] = np.array([1.0, 0.0, 0.0]) + 0.05 * rng.normal(size=d[::3].shape)
    d[::6] *= -1.0
    d /= np.linalg.norm(d, axis=1)[:, None]
    p0 = rng.uniform(0.0, 1.0, (m, 3)) * [10.0 * n, 16.0, 12.0] + [1.0, -8.0, -6.0]
    p0[::4, 0] = -rng.uniform(1.0, 9.0, p0[::4].shape[0])
    p1 = (p0 + d * L[:, None]).astype(np.float32).astype(np.float64)
    p0 = p0.astype(np.float32).astype(np.float64)
    for region, part in ((1, p0[:, 0] > 0), (0, p0[:, 0] < 0)):
        ou, onx, on = osc.find_end_of_step(region, p0[part], p1[part])
        gu, gnx, gn = pr.find_end_of_step(region, p0[part], p1[part])
        hit = ou <= 1.0
        assert hit.sum() > 100
        ok = (onx == gnx) & (hit == (gu <= 1.0))
        ok[hit] &= np.abs(ou[hit] - gu[hit]) * L[part][hit] < 1e-3
        # the last crossing of a segment that ends on a face may round either way
        assert np.sum(~ok) <= 3, (region, np.sum(~ok))
        both = ok & hit
        far = np.sort(np.abs(np.abs(on[both]) - 1.0), axis=1)[:, 0] < 1e-6   # not on an edge
        assert np.array_equal(on[both][far], gn[both][far].astype(np.float64))
