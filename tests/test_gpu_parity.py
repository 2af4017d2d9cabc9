"""GPU parity: libnbody_hip.so (through its C ABI) against the CPU oracle.

Bars: FP64 paths bit-exact (forces, integrator, octree sums); topology and
body order bit-exact; FP32 paths within stated relative tolerances against
the FP64 direct sum.
"""
import math

import numpy as np
import pytest

from helpers import assert_canonical_equal, clustered, rel_err, uniform_cube

pytestmark = pytest.mark.gpu


def star_disk(nb, n, seed=0x4E424F44590000):
    return nb.gen_star_disk(n, seed)


def plummer(nb, n, seed=0x4E424F44590002):
    return nb.gen_plummer(n, seed)


def make(gpu, kind, n, seed=1):
    if kind == "cube":
        return uniform_cube(n, seed)
    if kind == "cluster":
        return clustered(n, seed)
    if kind == "disk":
        return star_disk(gpu, n)
    if kind == "plummer":
        return plummer(gpu, n)
    raise ValueError(kind)


def ctx_for(gpu, d, **kw):
    c = gpu.Context(len(d["x"]), **kw)
    c.set_state(d["x"], d["y"], d["z"], d["vx"], d["vy"], d["vz"], d["m"])
    return c


def bits(a):
    return np.asarray(a, dtype=np.float64).view(np.int64)


# ---- direct sum ---------------------------------------------------------------------
@pytest.mark.parametrize("kind,n", [("cube", 1), ("cube", 2), ("cube", 65), ("cube", 1000),
                                    ("disk", 4099), ("cluster", 3000)])
def test_direct_f64_bitexact(gpu, oracle, kind, n):
    d = make(gpu, kind, n)
    with ctx_for(gpu, d) as c:
        ax, ay, az = c.forces_direct()
    rx, ry, rz = oracle.naive_accel(d["x"], d["y"], d["z"], d["m"])
    for a, r in ((ax, rx), (ay, ry), (az, rz)):
        np.testing.assert_array_equal(bits(a), bits(r))


def test_direct_targets_f64(gpu, oracle):
    d = make(gpu, "disk", 5000)
    t = np.array([0, 1, 4999, 2500, 17, 17], dtype=np.uint32)
    with ctx_for(gpu, d) as c:
        ax, ay, az = c.forces_direct_targets(t)
    rx, ry, rz = oracle.naive_accel_targets(d["x"], d["y"], d["z"], d["m"], t)
    for a, r in ((ax, rx), (ay, ry), (az, rz)):
        np.testing.assert_array_equal(bits(a), bits(r))


@pytest.mark.parametrize("kind,n,med,worst", [("disk", 16384, 1e-6, 1e-4),
                                              ("plummer", 20000, 1e-5, 1e-3),
                                              ("cube", 777, 1e-5, 1e-3)])
def test_direct_f32c_accuracy(gpu, oracle, kind, n, med, worst):
    d = make(gpu, kind, n)
    with ctx_for(gpu, d, precision=gpu.PREC_FP32C) as c:
        ax, ay, az = c.forces_direct()
    rx, ry, rz = oracle.naive_accel(d["x"], d["y"], d["z"], d["m"])
    e = rel_err(ax, ay, az, rx, ry, rz)
    assert np.median(e) < med, np.median(e)
    assert np.quantile(e, 0.999) < worst, np.quantile(e, 0.999)


def term_sum(d, G, eps2):
    """S_i = G sum_j m_j / (r_ij^2 + eps^2): the sum of the pair terms'
    magnitudes, the scale of a summation's rounding error."""
    x, y, z, m = (np.asarray(d[k], dtype=np.float64) for k in ("x", "y", "z", "m"))
    n = x.size
    S = np.empty(n)
    for i in range(0, n, 512):
        sl = slice(i, min(n, i + 512))
        r2 = (x[sl, None] - x) ** 2 + (y[sl, None] - y) ** 2 + (z[sl, None] - z) ** 2 + eps2
        t = m[None, :] / r2
        t[np.arange(sl.stop - sl.start), np.arange(sl.start, sl.stop)] = 0.0  # no self term
        S[sl] = G * t.sum(axis=1)
    return S


@pytest.mark.parametrize("kind,n", [("disk", 16384), ("plummer", 5000), ("cube", 1000),
                                    ("cluster", 3001), ("cube", 2), ("cube", 1)])
def test_direct_f64_fast_tolerance(gpu, oracle, kind, n):
    # FP64 pairs with the corrected v_rsq_f64 estimate, split sums added in a
    # fixed order.  Bounds: per body ||a - a_ref|| <= 1e-12 S_i (S_i above)
    # against the reference arithmetic, and a median error against a
    # long-double sum at most twice that of the reference arithmetic.
    d = make(gpu, kind, n)
    with ctx_for(gpu, d, precision=gpu.PREC_FP64_FAST) as c:
        ax, ay, az = c.forces_direct()
        again = c.forces_direct()
    for u, v in zip((ax, ay, az), again):
        np.testing.assert_array_equal(bits(u), bits(v))  # deterministic
    rx, ry, rz = oracle.naive_accel(d["x"], d["y"], d["z"], d["m"])
    diff = np.sqrt((ax - rx) ** 2 + (ay - ry) ** 2 + (az - rz) ** 2)
    S = term_sum(d, oracle.G_ref(), oracle.eps2_ref())
    assert np.all(diff <= 1e-12 * S), (diff / np.where(S > 0, S, 1)).max()
    if n > 1:
        # against a long-double sum on sampled targets: no worse than the
        # reference arithmetic itself (whose error here comes from partly
        # cancelling near-neighbour terms), up to a factor 2
        t = np.random.default_rng(0).choice(n, min(n, 256), replace=False)
        L = np.longdouble
        X, Y, Z, M = (np.asarray(d[k]).astype(L) for k in ("x", "y", "z", "m"))
        e_fast, e_ref = [], []
        for i in t:
            dx, dy, dz = X - X[i], Y - Y[i], Z - Z[i]
            r2 = dx * dx + dy * dy + dz * dz + L(oracle.eps2_ref())
            w = M / (r2 * np.sqrt(r2))
            w[i] = 0
            tx, ty, tz = (np.sum(w * c) * L(oracle.G_ref()) for c in (dx, dy, dz))
            nt = np.sqrt(tx * tx + ty * ty + tz * tz)
            for got, out in (((ax[i], ay[i], az[i]), e_fast), ((rx[i], ry[i], rz[i]), e_ref)):
                g = [L(v) for v in got]
                out.append(float(np.sqrt((g[0] - tx) ** 2 + (g[1] - ty) ** 2 + (g[2] - tz) ** 2)
                                 / nt))
        mf, mr = float(np.median(e_fast)), float(np.median(e_ref))
        print(f"median error vs long double: fast {mf:.3e}, reference arithmetic {mr:.3e}")
        assert mf <= max(2 * mr, 1e-15), (mf, mr)


# Both kernels of the bit-exact sum (16 and 64 targets per workgroup, chosen by
# the target count) at the edges of a workgroup's targets and of a chunk of
# sources (60 and 48), and on both sides of the rule between them (13,653 and
# 16,384 targets).  The second system has every other pair's term outside the
# range of the short IEEE sequences.
@pytest.mark.parametrize("n", [2, 15, 16, 17, 48, 49, 59, 60, 61, 121, 13652, 13655, 16385])
def test_direct_f64_kernels_bitexact(gpu, oracle, n):
    for scale in (1.0, 2.0 ** 90):
        if scale > 1 and n > 200:
            continue
        d = uniform_cube(n, 200 + n)
        d["x"][::2] *= scale
        with ctx_for(gpu, d) as c:
            got = c.forces_direct()
            t = np.arange(n - 1, -1, -1, dtype=np.uint32)[:300]
            sel = c.forces_direct_targets(t)
        ref = oracle.naive_accel(d["x"], d["y"], d["z"], d["m"])
        for g, s_, r in zip(got, sel, ref):
            np.testing.assert_array_equal(bits(g), bits(r))
            np.testing.assert_array_equal(bits(s_), bits(r[t]))


@pytest.mark.parametrize("n", [3, 63, 64, 65, 128, 129, 256, 257, 1024, 1025, 8191, 16383, 16385])
def test_direct_split_edges(gpu, oracle, n):
    # The split sums at the edges of a block's targets (64, 128), a wave's stage
    # (64) and run (256), a block's sources (256, 1024) and the changes of the
    # split rules (8192, 16,384).
    # FP64: 1e-12 S_i as above.  FP32, with positions that are FP32 numbers: a
    # term's relative error is at most about 20 roundings (r^2 5, raised to
    # -3/2, v_rsq_f32 1 ulp three times, the products) and a run adds 256 terms
    # before it is folded into FP64: 276 roundings, bound 512 * 2^-24 S_i.
    d = uniform_cube(n, 100 + n)
    for k in "xyz":
        d[k] = d[k].astype(np.float32).astype(np.float64)
    rx, ry, rz = oracle.naive_accel(d["x"], d["y"], d["z"], d["m"])
    S = term_sum(d, oracle.G_ref(), oracle.eps2_ref())
    for precision, bound in ((gpu.PREC_FP64_FAST, 1e-12), (gpu.PREC_FP32C, 512 * 2.0 ** -24)):
        with ctx_for(gpu, d, precision=precision) as c:
            ax, ay, az = c.forces_direct()
        diff = np.sqrt((ax - rx) ** 2 + (ay - ry) ** 2 + (az - rz) ** 2)
        assert np.all(diff <= bound * S), (precision, (diff / S).max())


# ratio: the bound on quadrupole error / monopole error.  The star + disk sits
# at the FP32 rounding floor (~9e-8, the star's force dominates), where cell
# expansions change nothing: there the quadrupole must only not be worse.
@pytest.mark.parametrize("kind,n,theta,ratio", [("plummer", 30000, 0.6, 0.5),
                                                 ("plummer", 30000, 0.9, 0.6),
                                                 ("cluster", 20000, 0.7, 0.6),
                                                 ("disk", 30000, 0.8, 1.05)])
def test_bh_quadrupole_accuracy(gpu, oracle, kind, n, theta, ratio):
    # Cells with their quadrupole moments: the same walk, octree and
    # interaction counts as monopole cells, and a median error against the
    # FP64 direct sum well below the monopole's at the same theta (the
    # quadrupole removes the leading (e/d)^2 term of the monopole's error and
    # leaves the octupole's (e/d)^3, so the ratio falls with theta: measured
    # 0.35 at theta 0.6 and 0.46 at 0.9 on the Plummer sphere; a wrong sign or
    # a dropped term raises the error above the monopole's).
    d = make(gpu, kind, n)
    rx, ry, rz = oracle.naive_accel(d["x"], d["y"], d["z"], d["m"])
    res = {}
    for quad in (0, 1):
        with ctx_for(gpu, d, theta=theta, precision=gpu.PREC_FP32C, quadrupole=quad) as c:
            c.bh_build()
            ax, ay, az = c.bh_forces()
            inter = c.interactions()
            qp = c.quadrupole_pairs()
        res[quad] = (np.median(rel_err(ax, ay, az, rx, ry, rz)), inter, qp)
    (e_m, i_m, q_m), (e_q, i_q, q_q) = res[0], res[1]
    print(f"{kind} theta {theta}: monopole {e_m:.3e}, quadrupole {e_q:.3e}, "
          f"{q_q / n:.0f} quadrupole cells per body of {i_q.mean():.0f}")
    np.testing.assert_array_equal(i_m, i_q)
    assert q_m == 0 and 0 < q_q < i_q.sum()
    assert e_q < ratio * e_m, (e_q, e_m)


def test_rsq_f64_newton_accuracy(gpu):
    # The inverse square root of the fast FP64 sum, checked on two bodies:
    # a(0) = G m1 r / (r^2 + eps^2)^(3/2) over a sweep of separations spanning
    # 1e-10 .. 1e10 AU, against the closed form in long double.
    G, eps2 = 1.0, 1e-22
    worst = 0.0
    for r in np.logspace(-10, 10, 41):
        d = dict(x=np.array([0.0, r]), y=np.zeros(2), z=np.zeros(2), vx=np.zeros(2),
                 vy=np.zeros(2), vz=np.zeros(2), m=np.array([1.0, 3.0]))
        with ctx_for(gpu, d, precision=gpu.PREC_FP64_FAST, G=G, eps2=eps2) as c:
            ax, _, _ = c.forces_direct()
        rl = np.longdouble(r)
        want = np.longdouble(3.0) * rl / (rl * rl + np.longdouble(eps2)) ** np.longdouble(1.5)
        worst = max(worst, float(abs((np.longdouble(ax[0]) - want) / want)))
    assert worst < 4e-15, worst


# ---- integrator -----------------------------------------------------------------------
def test_leapfrog_bitexact(gpu, oracle):
    d = make(gpu, "cube", 3001, 5)
    dt = 1.0 / 24
    with ctx_for(gpu, d) as c:
        c.forces_direct()
        a = c.accel()
        c.kick_drift(dt)
        s1 = c.state()
        c.forces_direct()
        a2 = c.accel()
        c.kick(dt)
        s2 = c.state()
    x = [d["x"].copy(), d["y"].copy(), d["z"].copy()]
    vh = oracle.kick_drift(dt, list(a), [d["vx"], d["vy"], d["vz"]], x)
    for k, ref in zip(("x", "y", "z"), x):
        np.testing.assert_array_equal(bits(s1[k]), bits(ref))
    v = oracle.kick(dt, list(a2), vh)
    for k, ref in zip(("vx", "vy", "vz"), v):
        np.testing.assert_array_equal(bits(s2[k]), bits(ref))


# ---- octree -----------------------------------------------------------------------------
def test_tree_reference_fixture(gpu, oracle):
    # tests/BarnesHutTest.cpp:11-33 and :75-127
    d = dict(x=np.array([0.0, 0.0, 2.0]), y=np.array([1.0, 0.0, 0.0]), z=np.array([0.0, 2.0, 0.0]),
             vx=np.zeros(3), vy=np.zeros(3), vz=np.zeros(3), m=np.array([10.0, 10.0, 10.0]))
    with ctx_for(gpu, d) as c:
        c.bh_build()
        info = c.tree_info()
        assert list(info["aabb"]) == [0, -0.5, 0, 2, 1.5, 2, 2]
        assert info["node_count"] == 9
        assert list(c.tree_sorted()) == [1, 2, 0]
        can = c.tree_canonical()
    assert can["mass"][0] == 30.0
    # body0 in digit 5, body2 in digit 3, body1 in digit 0
    kids = {int(can["body"][i]): i - 1 for i in range(1, 9) if can["kind"][i] == 1}
    assert kids == {0: 5, 2: 3, 1: 0}
    t = oracle.Tree(3, 48)
    t.build(d["x"], d["y"], d["z"], d["m"])
    assert_canonical_equal(can, t.canonical(), "fixture")


def test_tree_parity_repeated_builds(gpu, oracle):
    # The radix sort keeps control words (digit totals, tile counters, look-back
    # status) in the context between builds; three builds of different
    # positions on one context, 18 sort tiles each, must each match the oracle.
    n = 70001
    with gpu.Context(n) as c:
        for seed in (11, 12, 13):
            d = clustered(n, seed) if seed != 12 else uniform_cube(n, seed)
            c.set_state(d["x"], d["y"], d["z"], d["vx"], d["vy"], d["vz"], d["m"])
            c.bh_build()
            sorted_gpu = c.tree_sorted()
            can = c.tree_canonical()
            t = oracle.Tree(n)
            t.build(d["x"], d["y"], d["z"], d["m"])
            np.testing.assert_array_equal(sorted_gpu, t.export()["sorted"], err_msg=f"seed {seed}")
            assert_canonical_equal(can, t.canonical(), f"seed {seed}")


def test_tree_sort_more_tiles_than_resident(gpu, oracle):
    # 367 sort tiles of 8192 keys (the last one ragged; sorts of 2^21 keys and
    # more take the larger tiles, one block per CU): more tiles than the
    # device holds at once, so some look-back waits name tiles whose blocks
    # start later.  Two builds, positions moved in between.
    n = 3000017
    d = plummer(gpu, n)
    with ctx_for(gpu, d, precision=gpu.PREC_FP32C) as c:
        for step in range(2):
            if step:
                rng = np.random.default_rng(5)
                for k in ("x", "y", "z"):
                    d[k] = d[k] + rng.normal(0.0, 1e-3, n)
                c.set_positions(d["x"], d["y"], d["z"])
            c.bh_build()
            sorted_gpu = c.tree_sorted()
            info = c.tree_info()
            t = oracle.Tree(n)
            t.build(d["x"], d["y"], d["z"], d["m"])
            np.testing.assert_array_equal(sorted_gpu, t.export()["sorted"], err_msg=f"build {step}")
            assert info["node_count"] == t.node_count
            if step == 0:
                # centre-of-mass sums over 733 blocks of 2048 bodies and 23
                # super-blocks of 32 blocks
                assert_canonical_equal(c.tree_canonical(), t.canonical(), "3M plummer")


def test_tree_more_scan_tiles_than_read_inline(gpu, oracle):
    # 4,097 scan tiles of pairs and 4,098 of bodies: above 4,096 the tile sums are
    # scanned by a launch of their own, for the cells' numbers and the groups' places.
    # Every body must be in one group: its interactions are counted and its force
    # is near the direct sum's (opening angle 0.7: about 1e-3 in the median).
    n = 8390657
    d = plummer(gpu, n)
    t = oracle.Tree(n)
    t.build(d["x"], d["y"], d["z"], d["m"])
    with ctx_for(gpu, d, precision=gpu.PREC_FP32C, theta=0.7) as c:
        c.bh_build()
        np.testing.assert_array_equal(c.tree_sorted(), t.export()["sorted"])
        assert c.tree_info()["node_count"] == t.node_count
        a = c.bh_forces()
        assert np.all(c.interactions() > 0)
        sample = np.linspace(0, n - 1, 512).astype(np.uint32)
        ref = c.forces_direct_targets(sample)
    norm = np.sqrt(sum(r ** 2 for r in ref))
    err = np.sqrt(sum((g[sample] - r) ** 2 for g, r in zip(a, ref))) / norm
    assert np.median(err) < 3e-3, np.median(err)
    assert np.percentile(err, 99) < 0.05, np.percentile(err, 99)


def test_tree_sort_wide_tiles(gpu, oracle):
    # 207 sort tiles of 10,240 keys, the last one ragged: the size at which tiles
    # of 8192 keys would need a second round
    n = 2110001
    d = plummer(gpu, n)
    t = oracle.Tree(n)
    t.build(d["x"], d["y"], d["z"], d["m"])
    with ctx_for(gpu, d, precision=gpu.PREC_FP32C) as c:
        for _ in range(2):
            c.bh_build()
            np.testing.assert_array_equal(c.tree_sorted(), t.export()["sorted"])
        assert c.tree_info()["node_count"] == t.node_count


def test_tree_parity_deep_clusters(gpu, oracle):
    # 40 clumps of 3000 bodies, 1e-9 across (about 31 levels below the root):
    # every clump holds a block boundary, so each brings a chain of about 31
    # cells crossing it.  A super-block of 32 blocks then holds more such
    # cells than one workgroup sums in LDS (the global-memory path), while
    # the cells crossing the super-block boundary take the LDS path.
    rng = np.random.default_rng(21)
    k, per = 40, 3000
    centres = rng.uniform(-1, 1, (k, 3))
    p = (centres[:, None, :] + rng.uniform(-5e-10, 5e-10, (k, per, 3))).reshape(-1, 3)
    n = k * per
    d = dict(x=p[:, 0].copy(), y=p[:, 1].copy(), z=p[:, 2].copy(), vx=np.zeros(n),
             vy=np.zeros(n), vz=np.zeros(n), m=rng.uniform(1e20, 1e22, n))
    with ctx_for(gpu, d) as c:
        c.bh_build()
        info = c.tree_info()
        can = c.tree_canonical()
        srt = c.tree_sorted()
    assert info["max_depth"] > 30
    t = oracle.Tree(n)
    t.build(d["x"], d["y"], d["z"], d["m"])
    np.testing.assert_array_equal(srt, t.export()["sorted"])
    assert_canonical_equal(can, t.canonical(), "deep clusters")


@pytest.mark.parametrize("kind,n", [("cube", 1), ("cube", 2), ("cube", 9), ("cube", 1000),
                                    ("cluster", 5000), ("disk", 20000), ("plummer", 20000),
                                    ("cube", 70001)])
def test_tree_parity(gpu, oracle, kind, n):
    d = make(gpu, kind, n, seed=n)
    with ctx_for(gpu, d) as c:
        c.bh_build()
        info = c.tree_info()
        sorted_gpu = c.tree_sorted()
        can = c.tree_canonical()
    t = oracle.Tree(n)
    t.build(d["x"], d["y"], d["z"], d["m"])
    np.testing.assert_array_equal(info["aabb"], t.aabb)
    assert info["node_count"] == t.node_count
    np.testing.assert_array_equal(sorted_gpu, t.export()["sorted"])
    assert_canonical_equal(can, t.canonical(), f"{kind} n={n}")


# Edges of the build's blocks: 256 and 1024 bodies (topology, centre of mass),
# 2048 (scan), 4096 (sort), 64 blocks of 1024 (super-blocks: one body over, and a
# second super-block of two blocks).  Sums are the reference's, bit for bit.
@pytest.mark.parametrize("kind,n", [("cube", 3), ("cube", 255), ("plummer", 257),
                                    ("plummer", 1023), ("disk", 1024), ("cluster", 1025),
                                    ("plummer", 2047), ("cube", 2049), ("disk", 4095),
                                    ("cluster", 4096), ("plummer", 4097), ("cluster", 65536),
                                    ("plummer", 65537), ("disk", 66561)])
def test_tree_block_edges(gpu, oracle, kind, n):
    d = make(gpu, kind, n, seed=n)
    t = oracle.Tree(n)
    t.build(d["x"], d["y"], d["z"], d["m"])
    with ctx_for(gpu, d) as c:
        c.bh_build()
        assert c.tree_info()["node_count"] == t.node_count
        np.testing.assert_array_equal(c.tree_sorted(), t.export()["sorted"])
        assert_canonical_equal(c.tree_canonical(), t.canonical(), f"{kind} n={n}")


# Sorts by merging (runs of 2048 keys, then 16,384 and 131,072): a short last
# run, one key over, the largest such sort and the first by passes.  Bodies
# already in key order, and in its reverse, leave runs that do not overlap;
# "blocks" repeats a few positions' neighbourhoods so that one run's keys bound
# whole other runs (more keys between the bounds than fit the LDS).
@pytest.mark.parametrize("kind,n,order", [("plummer", 16384, "input"), ("cube", 16385, "input"),
                                          ("plummer", 20480, "sorted"), ("cube", 34000, "reversed"),
                                          ("plummer", 50001, "blocks"),
                                          ("plummer", 131329, "blocks"),
                                          ("disk", 262144, "input"), ("cube", 262145, "reversed")])
def test_tree_merge_sort_edges(gpu, oracle, kind, n, order):
    d = make(gpu, kind, n, seed=n)
    t = oracle.Tree(n)
    t.build(d["x"], d["y"], d["z"], d["m"])
    perm = np.arange(n)
    if order != "input":
        perm = np.asarray(t.export()["sorted"]).astype(np.int64)
        if order == "reversed":
            perm = perm[::-1]
        elif order == "blocks":  # every third run thinly spread, the others dense
            thin = perm[::3]
            rest = np.setdiff1d(perm, thin, assume_unique=True)
            perm = np.concatenate([rest[:n // 2], thin, rest[n // 2:]])
        d = {k: np.ascontiguousarray(v[perm]) for k, v in d.items()}
        t = oracle.Tree(n)
        t.build(d["x"], d["y"], d["z"], d["m"])
    with ctx_for(gpu, d) as c:
        for _ in range(2):
            c.bh_build()
            np.testing.assert_array_equal(c.tree_sorted(), t.export()["sorted"])
        assert_canonical_equal(c.tree_canonical(), t.canonical(), f"{kind} n={n} {order}")


def test_tree_deep_runs(gpu, oracle):
    # pairs of bodies closer than edge/2^21 force the 42-digit path
    rng = np.random.default_rng(3)
    n = 600
    base = rng.uniform(-1, 1, (n // 2, 3))
    off = rng.normal(0, 1e-9, (n // 2, 3))
    p = np.concatenate([base, base + off])
    d = dict(x=p[:, 0].copy(), y=p[:, 1].copy(), z=p[:, 2].copy(), vx=np.zeros(n),
             vy=np.zeros(n), vz=np.zeros(n), m=rng.uniform(1, 2, n))
    # ~25 single-child levels per pair: more nodes than the default 16*N storage
    with ctx_for(gpu, d, storage_size_param=512) as c:
        c.bh_build()
        info = c.tree_info()
        can = c.tree_canonical()
        srt = c.tree_sorted()
    assert info["max_depth"] > 21
    t = oracle.Tree(n, 512 * n)
    t.build(d["x"], d["y"], d["z"], d["m"])
    np.testing.assert_array_equal(srt, t.export()["sorted"])
    assert_canonical_equal(can, t.canonical(), "deep runs")


# ---- Barnes-Hut forces -------------------------------------------------------------------
# theta = 0 opens every cell, so the register batches of unvisited children
# spill to the memory stack on every level; n = 1 and 2 walk a root leaf and
# a root with two body leaves
@pytest.mark.parametrize("kind,n,theta", [("cube", 1, 0.5), ("cube", 2, 0.5), ("cube", 2000, 0.5),
                                          ("cube", 300, 0.0), ("cluster", 3000, 0.0),
                                          ("cluster", 4000, 1.05), ("disk", 20000, 0.5),
                                          ("plummer", 20000, 0.7)])
def test_bh_exact_bitexact(gpu, oracle, kind, n, theta):
    d = make(gpu, kind, n, seed=7)
    with ctx_for(gpu, d, theta=theta) as c:
        c.bh_build()
        ax, ay, az = c.bh_forces()
        inter = c.interactions()
    t = oracle.Tree(n)
    t.build(d["x"], d["y"], d["z"], d["m"])
    rx, ry, rz, rint = t.bh_accel(theta)
    np.testing.assert_array_equal(inter, rint)
    for a, r in ((ax, rx), (ay, ry), (az, rz)):
        np.testing.assert_array_equal(bits(a), bits(r))


# The two kernels of the bit-exact traversal: teams of eight lanes at the edges
# of a wave's bodies (8) and a workgroup's (32), waves of 64 bodies on both sides
# of the rule between them (100,000 bodies at theta 0.5, 210,000 at 1.05), whole
# waves and one body over.  theta 1e-150 and 1e150 leave the range in which the
# opening test is decided from squares.
@pytest.mark.parametrize("kind,n,theta", [("cube", 7, 0.5), ("cube", 8, 0.3), ("cube", 9, 0.0),
                                          ("cube", 31, 0.7), ("plummer", 33, 0.7),
                                          ("plummer", 65, 1e-150), ("plummer", 700, 1e150),
                                          ("plummer", 99999, 0.5), ("plummer", 100001, 0.5),
                                          ("cluster", 100032, 0.5), ("disk", 140033, 0.7),
                                          ("plummer", 209999, 1.05), ("disk", 210049, 1.05),
                                          ("plummer", 100001, 1e150)])
def test_bh_exact_kernels_bitexact(gpu, oracle, kind, n, theta):
    d = make(gpu, kind, n, seed=17)
    t = oracle.Tree(n)
    t.build(d["x"], d["y"], d["z"], d["m"])
    rx, ry, rz, rint = t.bh_accel(theta)
    for sort_bodies in (1, 0):
        with ctx_for(gpu, d, theta=theta, sort_bodies=sort_bodies) as c:
            c.bh_build()
            ax, ay, az = c.bh_forces()
            inter = c.interactions()
        np.testing.assert_array_equal(inter, rint)
        for a, r in ((ax, rx), (ay, ry), (az, rz)):
            np.testing.assert_array_equal(bits(a), bits(r))


# Both sides of the rule between the two kernels at larger opening angles: 170,000
# bodies from theta 0.85 on.
@pytest.mark.parametrize("kind,n,theta", [("plummer", 169999, 0.85), ("disk", 170017, 0.85),
                                          ("disk", 169991, 1.05), ("plummer", 170033, 1.4)])
def test_bh_exact_kernel_rule_bitexact(gpu, oracle, kind, n, theta):
    d = make(gpu, kind, n, seed=23)
    t = oracle.Tree(n)
    t.build(d["x"], d["y"], d["z"], d["m"])
    rx, ry, rz, rint = t.bh_accel(theta)
    with ctx_for(gpu, d, theta=theta) as c:
        c.bh_build()
        ax, ay, az = c.bh_forces()
        inter = c.interactions()
    np.testing.assert_array_equal(inter, rint)
    for a, r in ((ax, rx), (ay, ry), (az, rz)):
        np.testing.assert_array_equal(bits(a), bits(r))


def test_bh_exact_deep_runs(gpu, oracle):
    # pairs closer than edge/2^21: each pair hangs under ~25 single-child
    # cells, so the walk opens long chains whose pushed batches are all empty
    rng = np.random.default_rng(5)
    n = 600
    base = rng.uniform(-1, 1, (n // 2, 3))
    off = rng.normal(0, 1e-9, (n // 2, 3))
    p = np.concatenate([base, base + off])
    d = dict(x=p[:, 0].copy(), y=p[:, 1].copy(), z=p[:, 2].copy(), vx=np.zeros(n),
             vy=np.zeros(n), vz=np.zeros(n), m=rng.uniform(1, 2, n))
    for theta in (0.5, 0.0):
        with ctx_for(gpu, d, storage_size_param=512, theta=theta) as c:
            c.bh_build()
            ax, ay, az = c.bh_forces()
            inter = c.interactions()
        t = oracle.Tree(n, 512 * n)
        t.build(d["x"], d["y"], d["z"], d["m"])
        rx, ry, rz, rint = t.bh_accel(theta)
        np.testing.assert_array_equal(inter, rint)
        for a, r in ((ax, rx), (ay, ry), (az, rz)):
            np.testing.assert_array_equal(bits(a), bits(r))


@pytest.mark.parametrize("kind,n,theta", [("disk", 30000, 0.5), ("plummer", 30000, 0.5),
                                          ("plummer", 30000, 1.0), ("cluster", 8000, 0.7)])
def test_bh_group_accuracy(gpu, oracle, kind, n, theta):
    d = make(gpu, kind, n, seed=9)
    with ctx_for(gpu, d, theta=theta, precision=gpu.PREC_FP32C) as c:
        c.bh_build()
        ax, ay, az = c.bh_forces()
    rx, ry, rz = oracle.naive_accel(d["x"], d["y"], d["z"], d["m"])
    e = rel_err(ax, ay, az, rx, ry, rz)
    t = oracle.Tree(n)
    t.build(d["x"], d["y"], d["z"], d["m"])
    bx, by, bz, _ = t.bh_accel(theta)
    eref = rel_err(bx, by, bz, rx, ry, rz)
    # opening a cell when any body of the group needs it is at least as
    # accurate as the per-body test; FP32 pair maths adds ~1e-6
    assert np.median(e) <= np.median(eref) + 2e-6, (np.median(e), np.median(eref))
    # the tail too: no body may be worse than the per-body traversal's worst
    # body by more than FP32 rounding
    assert np.quantile(e, 0.999) <= np.quantile(eref, 0.999) + 1e-5
    assert e.max() <= 2 * eref.max() + 1e-5, (e.max(), eref.max(), int(np.argmax(e)))
    if kind == "disk":
        # the star dominates every force: far below the 1e-4 bar
        assert np.median(e) < 1e-6


# ---- full loop ------------------------------------------------------------------------------
@pytest.mark.parametrize("algo", ["naive", "BarnesHut"])
def test_simulation_loop_bitexact(gpu, oracle, algo):
    n = 3000
    d = make(gpu, "disk", n)
    dt, steps = 1.0 / 24, 6
    theta = 0.5
    with ctx_for(gpu, d, theta=theta) as c:
        if algo == "naive":
            c.forces_direct()
        else:
            c.bh_build()
            c.bh_forces()
        c.steps(algo, dt, steps)
        s = c.state()
        a = c.accel()
    r = oracle.simulate(algo, d["x"], d["y"], d["z"], d["vx"], d["vy"], d["vz"], d["m"], dt,
                        steps * dt, theta=theta)
    assert r["steps"] == steps
    for k in ("x", "y", "z", "vx", "vy", "vz"):
        np.testing.assert_array_equal(bits(s[k]), bits(r[k]), err_msg=k)
    for got, k in zip(a, ("ax", "ay", "az")):
        np.testing.assert_array_equal(bits(got), bits(r[k]), err_msg=k)


def test_phase_times_are_nested_and_complete(gpu):
    """Phase timing: coinciding phase boundaries share one event.  Every phase
    of a Barnes-Hut run has a time, the build's sub-phases add up to at most
    the octree phase that holds them, and the keys and sort phases to at most
    "keys and sort"."""
    d = make(gpu, "disk", 200000)
    with ctx_for(gpu, d, theta=0.5, precision=gpu.PREC_FP32C) as c:
        c.bh_build()
        c.bh_forces()
        c.steps(gpu.ALGO_BARNES_HUT, 1.0 / 24, 3)
        ph = c.phase_ms()
    for k, v in ph.items():
        assert v > 0, (k, ph)
    sub = ph["AABB creation"] + ph["keys and sort"] + ph["topology"] + ph["Compute center of mass"]
    assert sub <= ph["Octree creation"] * 1.001 + 1e-3, ph
    assert ph["keys"] + ph["sort"] <= ph["keys and sort"] * 1.001 + 1e-3, ph


@pytest.mark.parametrize("algo", ["naive", "BarnesHut"])
def test_snapshot_async_matches_sync_reads(gpu, oracle, algo):
    # nb_snapshot_begin/wait return the state as it was at begin, although
    # further steps overwrite it while the DMA is in flight
    n = 5000
    d = make(gpu, "disk", n)
    dt, theta = 1.0 / 24, 0.5
    keys = ["x", "y", "z", "vx", "vy", "vz"]
    with ctx_for(gpu, d, theta=theta) as c:
        with pytest.raises(gpu.NBodyError):
            c.snapshot_wait()  # nothing begun yet
        if algo == "naive":
            c.forces_direct()
        else:
            c.bh_build()
            c.bh_forces()
        for rep in range(3):
            c.steps(algo, dt, 2)
            want, acc = c.state(), c.accel()
            c.snapshot_begin()
            c.steps(algo, dt, 3)
            got = c.snapshot_wait()
            for k in keys:
                np.testing.assert_array_equal(bits(got[k]), bits(want[k]), err_msg=f"{rep} {k}")
            for k, a in zip(("ax", "ay", "az"), acc):
                np.testing.assert_array_equal(bits(got[k]), bits(a), err_msg=f"{rep} {k}")
            if rep == 0:
                r = oracle.simulate(algo, d["x"], d["y"], d["z"], d["vx"], d["vy"], d["vz"],
                                    d["m"], dt, 2 * dt, theta=theta)
                for k in keys + ["ax", "ay", "az"]:
                    np.testing.assert_array_equal(bits(got[k]), bits(r[k]), err_msg=k)
        # a second begin before any wait: the wait returns the second state
        c.snapshot_begin()
        c.steps(algo, dt, 1)
        want = c.state()
        c.snapshot_begin()
        c.steps(algo, dt, 1)
        got = c.snapshot_wait()
        again = c.snapshot_wait()  # waiting twice returns the same snapshot
        for k in keys:
            np.testing.assert_array_equal(bits(got[k]), bits(want[k]), err_msg=k)
            np.testing.assert_array_equal(bits(again[k]), bits(want[k]), err_msg=k)


# ---- error handling ----------------------------------------------------------------------------
# State and accelerations read back at the edges of the copy paths (six arrays:
# one kernel up to 1 MiB, the runtime's copies up to 6 MiB, then chunks of
# 256 KiB, from 16 MiB on of 1 MiB; the last chunk of an array is short), twice,
# and with some of the arrays only.
@pytest.mark.parametrize("n", [1, 31, 33, 21845, 21846, 131071, 131073, 349525, 349527, 400001])
def test_state_read_back(gpu, n):
    rng = np.random.default_rng(n)
    keys = ("x", "y", "z", "vx", "vy", "vz", "m")
    d = {k: rng.normal(0, 1, n) for k in keys}
    with gpu.Context(n) as c:
        c.set_state(*[d[k] for k in keys])
        for _ in range(2):
            s = c.state()
            for k in keys[:6]:
                np.testing.assert_array_equal(s[k], d[k])
        y, vz = np.empty(n), np.empty(n)
        none = None
        assert c.lib.nb_get_state(c.h, none, y.ctypes.data_as(gpu._dp), none, none, none,
                                  vz.ctypes.data_as(gpu._dp)) == 0
        np.testing.assert_array_equal(y, d["y"])
        np.testing.assert_array_equal(vz, d["vz"])
        assert c.lib.nb_get_state(c.h, none, none, none, none, none, none) == 0
        c.kick_drift(0.0)
        assert all(np.all(a == 0) for a in c.accel())


# Accelerations read back at the edges of the copy paths (three arrays: one kernel up
# to 1.75 MiB, the runtime's copies up to 16 MiB, then chunks of 1 MiB), into memory
# that holds something else, against the snapshot, which takes another way.
@pytest.mark.parametrize("n", [2, 33, 21846, 30001, 76458, 76459, 349527, 699050, 699051, 800001])
def test_accel_read_back(gpu, n):
    d = plummer(gpu, n)
    with ctx_for(gpu, d, precision=gpu.PREC_FP32C, theta=1.0) as c:
        c.bh_build()
        assert c.lib.nb_bh_forces(c.h) == 0
        c.snapshot_begin()
        snap = c.snapshot_wait()
        for _ in range(2):
            got = [np.full(n, np.nan) for _ in range(3)]
            assert c.lib.nb_get_accel(c.h, *[g.ctypes.data_as(gpu._dp) for g in got]) == 0
            for g, k in zip(got, ("ax", "ay", "az")):
                np.testing.assert_array_equal(bits(g), bits(snap[k]))
                assert np.all(np.isfinite(g)) and np.any(g != 0)
        assert not np.array_equal(got[0], got[1]) and not np.array_equal(got[1], got[2])
        only = np.full(n, np.nan)
        assert c.lib.nb_get_accel(c.h, None, None, only.ctypes.data_as(gpu._dp)) == 0
        np.testing.assert_array_equal(bits(only), bits(snap["az"]))


def test_coincident_bodies_reported(gpu):
    d = uniform_cube(100, 2)
    d["x"][5], d["y"][5], d["z"][5] = d["x"][9], d["y"][9], d["z"][9]
    with ctx_for(gpu, d) as c:
        with pytest.raises(gpu.NBodyError) as e:
            c.bh_build()
        assert e.value.code == gpu.NB_E_DEPTH


def test_zero_mass_reported(gpu):
    d = uniform_cube(100, 3)
    d["m"][4] = 0.0
    with ctx_for(gpu, d) as c:
        with pytest.raises(gpu.NBodyError) as e:
            c.bh_build()
        assert e.value.code == gpu.NB_E_ZERO_MASS


def test_nan_position_reported(gpu):
    d = uniform_cube(100, 4)
    d["y"][50] = np.nan
    with ctx_for(gpu, d) as c:
        with pytest.raises(gpu.NBodyError) as e:
            c.bh_build()
        assert e.value.code == gpu.NB_E_AABB


def test_forces_before_build(gpu):
    d = uniform_cube(100, 5)
    with ctx_for(gpu, d) as c:
        with pytest.raises(gpu.NBodyError) as e:
            c.bh_forces()
        assert e.value.code == gpu.NB_E_NOT_BUILT


def test_storage_overflow_reported(gpu):
    d = clustered(4000, 6)
    with ctx_for(gpu, d, storage_size_param=1) as c:
        with pytest.raises(gpu.NBodyError) as e:
            c.bh_build()
        assert e.value.code == gpu.NB_E_NODE_OVERFLOW


@pytest.mark.parametrize("n,storage", [(4096, 1 << 20), (16, 1 << 31)])
def test_oversized_storage_keeps_context(gpu, n, storage):
    # storage_size_param * n beyond 2^29 nodes (the second case wraps a 32-bit
    # cell count to 0): rejected before any buffer is touched; the context
    # keeps its parameters and octree storage and builds as before
    d = uniform_cube(n, 7)
    with ctx_for(gpu, d, theta=0.5, precision=gpu.PREC_FP32C) as c:
        c.bh_build()
        want = c.bh_forces()
        with pytest.raises(gpu.NBodyError) as e:
            c.set_params(storage_size_param=storage)
        assert e.value.code == gpu.NB_E_INVALID_ARG
        assert c.params.storage_size_param == 16
        c.bh_build()
        got = c.bh_forces()
        # a valid change reallocates and still builds the same tree
        c.set_params(storage_size_param=24)
        c.bh_build()
        again = c.bh_forces()
    for u, v, w in zip(want, got, again):
        np.testing.assert_array_equal(bits(u), bits(v))
        np.testing.assert_array_equal(bits(u), bits(w))


# ---- full-size properties ------------------------------------------------------------------------
def test_million_body_tree_properties(gpu):
    n = 1 << 20
    d = make(gpu, "disk", n)
    with ctx_for(gpu, d, theta=0.5, precision=gpu.PREC_FP32C) as c:
        c.bh_build()
        info = c.tree_info()
        srt = c.tree_sorted()
        assert np.array_equal(np.sort(srt), np.arange(n, dtype=np.uint32))
        assert info["node_count"] == 1 + 8 * info["internal_count"]
        can = c.tree_canonical()
        assert can["count"][0] == n
        assert (can["kind"] == 1).sum() == n
        np.testing.assert_array_equal(can["body"][can["kind"] == 1], srt)
        ax, ay, az = c.bh_forces()
        rng = np.random.default_rng(0)
        t = np.sort(rng.choice(n, 16384, replace=False)).astype(np.uint32)
        rx, ry, rz = c.forces_direct_targets(t)
    e = rel_err(ax[t], ay[t], az[t], rx, ry, rz)
    assert np.median(e) < 1e-4


def test_plummer_4m_traversal_meets_the_error_bound(gpu):
    # The headline configuration at full size: 4,194,304-body Plummer sphere,
    # FP32 pairs with FP64 accumulation, at the opening angle bench.py picks
    # (0.36) and at theta 0.3.  Every body appears once in the octree order,
    # the node count is 1 + 8 * internal cells, and the median relative error
    # over 16,384 sampled targets against the FP64 direct sum (reference
    # arithmetic) is within 1e-4; a smaller theta is more accurate and costs
    # more interactions.
    n = 1 << 22
    d = gpu.gen_plummer(n, 0x4E424F44590002)
    t = np.sort(np.random.default_rng(1).choice(n, 16384, replace=False)).astype(np.uint32)
    res = {}
    with ctx_for(gpu, d, theta=0.36, precision=gpu.PREC_FP32C) as c:
        rx, ry, rz = c.forces_direct_targets(t)
        for theta in (0.36, 0.3):
            c.set_params(theta=theta)
            c.bh_build()
            srt = c.tree_sorted()
            assert np.array_equal(np.sort(srt), np.arange(n, dtype=np.uint32))
            info = c.tree_info()
            assert info["node_count"] == 1 + 8 * info["internal_count"]
            ax, ay, az = c.bh_forces()
            e = np.median(rel_err(ax[t], ay[t], az[t], rx, ry, rz))
            res[theta] = (e, c.interactions().mean())
            print(f"4M Plummer theta {theta}: median error {e:.3e}, "
                  f"{res[theta][1]:.0f} interactions per body")
    assert res[0.36][0] <= 1e-4 and res[0.3][0] < res[0.36][0]
    assert res[0.3][1] > res[0.36][1]


# ---- energy diagnostics ----------------------------------------------------------------
@pytest.mark.parametrize("kind,n", [("disk", 5000), ("cube", 777)])
def test_energy_bitexact(gpu, oracle, kind, n):
    d = make(gpu, kind, n)
    with ctx_for(gpu, d) as c:
        e = c.energy()
    r = oracle.energy(d["x"], d["y"], d["z"], d["vx"], d["vy"], d["vz"], d["m"])
    for k in ("kinetic", "potential", "total", "virial"):
        assert np.float64(e[k]).view(np.int64) == np.float64(r[k]).view(np.int64), k


# The energy kernels at the edges of a workgroup's bodies (64) and of a chunk of
# sources (48), with masses of which some take the plain operators (zero, and
# below 2^-150 of the unit), and on both sides of the rule between the two
# kernels (196,608 bodies; 768 and 769 blocks of rows, an odd round of them).
@pytest.mark.parametrize("n", [1, 2, 47, 48, 49, 63, 64, 65, 96, 97, 129, 20011, 196607, 196869])
def test_energy_edges_bitexact(gpu, oracle, n):
    d = uniform_cube(n, 300 + n)
    for k in range(3, n, 17):
        d["m"][k] = 0.0 if k % 2 else 1e-60
    with ctx_for(gpu, d) as c:
        e = c.energy()
    r = oracle.energy(d["x"], d["y"], d["z"], d["vx"], d["vy"], d["vz"], d["m"])
    for k in ("kinetic", "potential", "total"):
        assert np.float64(e[k]).view(np.int64) == np.float64(r[k]).view(np.int64), k


# The FP64 kernels take 1/sqrt(v) and a/sqrt(v) through the IEEE sequences
# without their range handling only for v (and a) inside fixed ranges
# (den^3 in [2^-512, 2^512] for the forces, v in [2^-600, 2^600] and |a| in
# [2^-300, 2^300] for the energy) and call the plain operators outside.  Two
# bodies per system, so that each pair term decides a result's bits on its
# own: separations on both sides of every bound, against the oracle.
@pytest.mark.parametrize("sep,m1", [(1e-40, 1.0), (1e-20, 1.0), (1.0, 1.0), (1e20, 1.0),
                                    (1e40, 1.0), (1e-100, 1.0), (1e100, 1.0),
                                    (1.0, 1e-60), (3e-10, 1e-70)])
def test_ieee_sequences_both_sides_of_their_range(gpu, oracle, sep, m1):
    d = dict(x=np.array([0.0, sep]), y=np.array([0.0, 0.5 * sep]), z=np.zeros(2),
             vx=np.array([1e-3, -2e-3]), vy=np.zeros(2), vz=np.zeros(2),
             m=np.array([m1, 2.5]))
    eps2 = 1e-90  # self terms stay finite (0 * 1/sqrt(eps2^3)); far below every d^2 here
    if sep < 1e-50:  # den^3 would underflow: forces only through the energy
        eps2 = None
    if eps2 is not None:
        with ctx_for(gpu, d, eps2=eps2) as c:
            ax, ay, az = c.forces_direct()
        rx, ry, rz = oracle.naive_accel(d["x"], d["y"], d["z"], d["m"], eps2=eps2)
        for a, r in ((ax, rx), (ay, ry), (az, rz)):
            assert np.all(np.isfinite(r))
            np.testing.assert_array_equal(bits(a), bits(r))
    with ctx_for(gpu, d) as c:
        e = c.energy()
    r = oracle.energy(d["x"], d["y"], d["z"], d["vx"], d["vy"], d["vz"], d["m"])
    for k in ("kinetic", "potential", "total"):
        assert np.float64(e[k]).view(np.int64) == np.float64(r[k]).view(np.int64), k


@pytest.mark.parametrize("n", [1, 2, 65, 2047, 2048, 2049, 4097])
def test_bh_group_list_edges(gpu, n):
    # the group list at the edges of its scan tiles (2048 positions): with
    # theta = 0 every body's list is every body, so a group missing or listed
    # twice at another place would leave a body out or count it differently
    d = make(gpu, "plummer", n, seed=n)
    with ctx_for(gpu, d, theta=0.0, precision=gpu.PREC_FP32C) as c:
        for _ in range(2):
            c.bh_build()
            ax = c.bh_forces()[0]
            np.testing.assert_array_equal(c.interactions(), np.full(n, n))
        assert np.all(np.isfinite(ax))


def _offset_of(d2):
    """dx, dy with dx^2 + dy^2 == d2 in FP64 (dx^2 exact)."""
    for m in range(1, 400):
        dx = math.floor(math.sqrt(d2) * 2.0**20) / 2.0**20 - m * 2.0**-20
        dy0 = math.sqrt(d2 - dx * dx)
        for w in range(-3, 4):
            dy = dy0 + w * math.ulp(dy0)
            if dx * dx + dy * dy == d2:
                return dx, dy
    return None


def test_inverse_root_of_ones(gpu, oracle):
    # roots whose significand is all ones, where the reciprocal's last step would
    # round the wrong way: 4 - 2^-50 and 4 - 2^-51 (times powers of four) as the
    # cubed squared distance of the force, and as the squared distance of the energy
    forces = energies = 0
    for k in range(-6, 7):
        for j in (1, 2):
            target = math.ldexp(4 - j * 2.0**-51, 2 * k)
            assert np.float64(math.sqrt(target)).view(np.int64) & (2**52 - 1) == 2**52 - 1
            c = target ** (1 / 3)
            roots = [c + t * math.ulp(c) for t in range(-60, 61)]
            cubes = [d for d in roots if (d * d) * d == target]
            for d2, energy in [(d, False) for d in cubes[:1]] + [(target, True)]:
                off = _offset_of(d2)
                if off is None:
                    continue
                d = dict(x=np.array([0.0, off[0]]), y=np.array([0.0, off[1]]), z=np.zeros(2),
                         vx=np.zeros(2), vy=np.zeros(2), vz=np.zeros(2), m=np.array([1.0, 2.0]))
                with ctx_for(gpu, d, theta=0.5) as ctx:
                    if energy:
                        e = ctx.energy()
                        r = oracle.energy(*(d[q] for q in ("x", "y", "z", "vx", "vy", "vz", "m")))
                        assert (np.float64(e["potential"]).view(np.int64)
                                == np.float64(r["potential"]).view(np.int64)), (k, j)
                        energies += 1
                        continue
                    direct = ctx.forces_direct()
                    ctx.bh_build()
                    walk = ctx.bh_forces()
                t = oracle.Tree(2)
                t.build(d["x"], d["y"], d["z"], d["m"])
                for got, want in ((direct, oracle.naive_accel(d["x"], d["y"], d["z"], d["m"])),
                                  (walk, t.bh_accel(0.5)[:3])):
                    for a, r in zip(got, want):
                        np.testing.assert_array_equal(bits(a), bits(r), err_msg=f"{k} {j}")
                forces += 1
    assert forces >= 4 and energies >= 20, (forces, energies)


def test_bh_forces_repeatable(gpu):
    # the traversal must not depend on state left by an earlier traversal of
    # the same octree (work-queue cursors, accumulators)
    d = make(gpu, "plummer", 20000)
    for prec in (gpu.PREC_FP32C, gpu.PREC_FP64):
        with ctx_for(gpu, d, theta=0.6, precision=prec) as c:
            c.bh_build()
            a1 = c.bh_forces()
            a2 = c.bh_forces()
        for u, v in zip(a1, a2):
            np.testing.assert_array_equal(bits(u), bits(v))
        assert np.all(np.isfinite(a1[0])) and np.abs(a1[0]).max() > 0


@pytest.mark.parametrize("group_max", [1, 5, 11, 13, 17, 22, 23, 26, 33, 40, 49, 53, 64])
def test_bh_group_passes_cover_every_pair(gpu, oracle, group_max):
    # theta = 0 opens every cell, so each group's list is every body of the
    # system and the traversal is an FP32 direct sum.  The group sizes span
    # one pass (1, 5, 64) and the two-pass splits of the flush (11 -> 3 + 8,
    # 13 -> 4 + 9, 17 -> 1 + 16, 22 -> 1 + 21, 40 -> 8 + 32, 53 -> 21 + 32, ...),
    # so a lane mapping that drops or repeats a share of the list shows as a
    # wrong interaction count or a force error far above FP32 rounding.
    n = 3000
    d = make(gpu, "cluster", n, seed=3)
    with ctx_for(gpu, d, theta=0.0, precision=gpu.PREC_FP32C, group_max=group_max,
                 pack_max=4 * group_max) as c:
        c.bh_build()
        ax, ay, az = c.bh_forces()
        inter = c.interactions()
    np.testing.assert_array_equal(inter, np.full(n, n, np.uint32))
    rx, ry, rz = oracle.naive_accel(d["x"], d["y"], d["z"], d["m"])
    e = rel_err(ax, ay, az, rx, ry, rz)
    # FP32 pairs summed in FP32 over at most 128 entries, folded into FP64; a
    # dropped or repeated share of the list would put most bodies near 1e-1
    assert np.median(e) < 1e-5, np.median(e)
    assert np.quantile(e, 0.999) < 1e-3, np.quantile(e, 0.999)
