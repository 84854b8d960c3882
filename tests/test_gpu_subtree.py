"""Trees whose nodes are at the limits of what one workgroup builds by itself:
its elements, its segments, the three lists together, nodes above the largest
node size down to single elements, more nodes than the passes hold in LDS, more
subtrees than their table, and coordinates that are not numbers.  Permutation,
leaves and lists against the oracle's, bit for bit."""
import numpy as np
import pytest

import vvflow_amd as V
from cases import cylinder_corners, oracle_for, path_code32
from test_gpu_heat import HEAT, STREAK, mirror

pytestmark = pytest.mark.gpu

DBL_MAX = np.finfo(np.float64).max


@pytest.fixture(scope="module")
def ctx():
    c = V.Context(0)
    yield c
    c.close()


def cloud(n, seed, spread=1.0):
    r = np.random.default_rng(seed)
    o = np.zeros((n, 6))
    o[:, :2] = r.uniform(-spread, spread, (n, 2)) ** 3
    o[:, 2] = r.choice([-1.0, 1.0], n) * r.uniform(0.5, 1.5, n) * 1e-3
    o[:, 3] = np.arange(n)   # the number travels with the record
    return o


def same_tree(ctx, o, tree):
    mirror(ctx, o)
    o.tree_build(*tree)
    ctx.tree_build(*tree)
    t = o.tree()
    lf = t["leaves"]
    g = ctx.tree_leaves()
    assert np.array_equal(g["geom"], t["geom"][lf], equal_nan=True)
    assert np.array_equal(g["ints"][:, :2], t["ints"][lf, :2])
    assert np.array_equal(g["ints"][:, 2:], t["ints"][lf, 4:6])   # depth, segments
    code = path_code32(t["path"])
    assert np.array_equal(path_code32(g["path"]), code[lf])
    depth = t["ints"][:, 4]
    assert np.array_equal(ctx.download()[:, 3], o.vortices()[:, 3])
    for lid in (HEAT, STREAK):
        assert np.array_equal(ctx.download_list(lid)[:, 3], o.get_list(lid)[:, 3])
    assert np.array_equal(ctx.tree_leaf_lists(), o.leaf_hs())
    for far in (False, True):
        g = ctx.tree_lists(far=far)
        off, nodes = t["far" if far else "near"]
        assert np.array_equal(g["off"], off)
        assert np.array_equal(path_code32(g["path"]), code[nodes])
        assert np.array_equal(g["depth"], depth[nodes])
        if far:
            cm = t["cm"][nodes]
            assert np.array_equal(g["cm"], cm, equal_nan=True)
    return len(lf), len(code)


# 1536 elements, 256 segments
@pytest.mark.parametrize("nv,nh,ns,nseg", [
    (1535, 0, 0, 0), (1536, 0, 0, 0), (1537, 0, 0, 0), (3072, 0, 0, 0), (3073, 0, 0, 0),
    (1, 0, 0, 0), (15, 15, 15, 15), (16, 0, 0, 3), (0, 1536, 0, 0), (0, 0, 1537, 0), (0, 17, 5, 0),
    (512, 512, 512, 0), (512, 512, 513, 0), (1000, 535, 1, 100), (5, 1500, 31, 40),
    (500, 0, 0, 255), (500, 0, 0, 256), (500, 0, 0, 257), (1280, 100, 156, 256), (1280, 100, 157, 256)])
def test_sizes_vs_oracle(ctx, nv, nh, ns, nseg):
    print(f"case subtree sizes {nv} {nh} {ns} segments {nseg}", flush=True)
    o = oracle_for(cloud(nv, 1), corners=cylinder_corners(nseg, 0.3) if nseg else None)
    o.set_list(HEAT, cloud(nh, 2))
    o.set_list(STREAK, cloud(ns, 3))
    same_tree(ctx, o, (8, 0.0, DBL_MAX))


# above the largest node size a node splits whatever it holds: 448 elements fit
@pytest.mark.parametrize("nv,nh,nseg", [(447, 0, 0), (448, 0, 0), (449, 0, 0), (224, 224, 0), (200, 200, 48), (200, 200, 49),
                                        (1536, 0, 0), (2000, 50, 60)])
@pytest.mark.parametrize("most", [1e-3, 0.2])
def test_small_largest_node_vs_oracle(ctx, nv, nh, nseg, most):
    print(f"case subtree largest node {most} {nv} {nh} segments {nseg}", flush=True)
    o = oracle_for(cloud(nv, 4), corners=cylinder_corners(nseg, 0.3) if nseg else None)
    o.set_list(HEAT, cloud(nh, 5))
    same_tree(ctx, o, (8, 0.0, most))


@pytest.mark.parametrize("per", [20, 45])
def test_more_nodes_than_the_passes_hold(ctx, per):
    """Clusters that halve towards a point split off one element a level: trees
    of about 900 and 2000 nodes over 1530 elements in one workgroup."""
    print(f"case subtree nodes, {per} a cluster", flush=True)
    k = 1530 // per
    o = cloud(k * per, 6)
    c, q = np.divmod(np.arange(k * per), per)
    o[:, 0] = 4.0 * (c % 8) + 2.0 ** -(q + 1.0)
    o[:, 1] = 4.0 * (c // 8) + 0.3 * 2.0 ** -(q + 1.0)
    leaves, nodes = same_tree(ctx, oracle_for(o), (8, 0.0, DBL_MAX))
    print(f"  {leaves} leaves, {nodes} nodes", flush=True)
    assert per < 45 or nodes > 1024


def leaves_of(x, y):
    """The tree's leaves (geometry, range) and order by its rules in plain numpy:
    boxes of the numbers there are, an element goes left only if it lies below
    the centre, and the k-th element left of the split that goes right trades
    places with the k-th from the end that goes left."""
    perm, out = np.arange(len(x)), []

    def box(a):
        a = a[~np.isnan(a)]
        return (a.min(), a.max()) if len(a) else (DBL_MAX, -DBL_MAX)

    def node(b, e):
        (lx, hx), (ly, hy) = box(x[perm[b:e]]), box(y[perm[b:e]])
        h, w, cx, cy = hy - ly, hx - lx, (lx + hx) * 0.5, (ly + hy) * 0.5
        if min(h, w) <= 0 or e - b < 16:
            out.append((cx, cy, h, w, b, e))
            return
        p = perm[b:e]
        left = x[p] < cx if h < w else y[p] < cy
        m = b + int(left.sum())
        a, z = b + np.flatnonzero(~left[:m - b]), m + np.flatnonzero(left[m - b:])[::-1]
        perm[a], perm[z] = perm[z], perm[a].copy()
        node(b, m)
        node(m, e)

    with np.errstate(over="ignore"):
        node(0, len(x))
    return perm, np.array(out)


@pytest.mark.parametrize("n", [40, 1536, 1537, 5000])
@pytest.mark.parametrize("numbers", [True, False])
def test_coordinates_that_are_no_numbers(ctx, n, numbers):
    """Elements without a number for a coordinate end in a leaf like the others
    and belong to no box (the reference's partition has no rule for them)."""
    print(f"case subtree NaN n={n} {numbers}", flush=True)
    v = cloud(n, 7)
    if not numbers:
        v[3::29, 0] = np.nan
        v[5::31, 1] = np.nan
        v[7::37, :2] = np.nan
    perm, ref = leaves_of(v[:, 0], v[:, 1])
    ctx.set_params(re=600.0, dt=0.005)
    ctx.upload_bodies(np.zeros(0, V.SEG_DTYPE), np.zeros(0, V.BODY_DTYPE))
    for lid in (HEAT, STREAK):
        ctx.upload_list(lid, np.zeros((0, 6)))
    ctx.upload(v)
    assert np.array_equal(ctx.tree_build(8, perm=True), perm)
    g = ctx.tree_leaves()
    assert np.array_equal(g["geom"], ref[:, :4])
    assert np.array_equal(g["ints"][:, :2], ref[:, 4:])


def test_more_subtrees_than_their_table(ctx):
    """Clumps of 225 elements above the largest node size: two do not fit a
    workgroup together, and 11264 of them are more than the table has room for.
    The tree's own properties (the oracle's lists would take minutes)."""
    print("case subtree table", flush=True)
    r = np.random.default_rng(8)
    gx, gy = np.meshgrid(np.arange(128), np.arange(88))
    c = np.repeat(np.stack([gx.ravel(), gy.ravel()], 1) * 3.0, 225, axis=0)
    v = np.zeros((len(c), 6))
    v[:, :2] = c + r.uniform(0, 1, c.shape)
    v[:, 2] = 1e-3
    perm0 = r.permutation(len(v))
    v = v[perm0]
    ctx.set_params(re=600.0, dt=0.005)
    ctx.upload_bodies(np.zeros(0, V.SEG_DTYPE), np.zeros(0, V.BODY_DTYPE))
    for lid in (HEAT, STREAK):
        ctx.upload_list(lid, np.zeros((0, 6)))
    ctx.upload(v)
    perm = ctx.tree_build(8, 0.0, 0.5, perm=True)
    assert np.array_equal(np.sort(perm), np.arange(len(v)))
    w = ctx.download()
    assert np.array_equal(w[:, :2], v[perm, :2])
    lv = ctx.tree_leaves()
    b, e = lv["ints"][:, 0], lv["ints"][:, 1]
    assert b[0] == 0 and e[-1] == len(v) and np.array_equal(b[1:], e[:-1]) and np.all(e > b)
    lo = np.stack([np.minimum.reduceat(w[:, k], b) for k in (0, 1)], 1)
    hi = np.stack([np.maximum.reduceat(w[:, k], b) for k in (0, 1)], 1)
    assert np.array_equal(lv["geom"][:, :2], (lo + hi) * 0.5)
    assert np.array_equal(lv["geom"][:, 2:], (hi - lo)[:, ::-1])   # h, w
    big = np.maximum(hi[:, 0] - lo[:, 0], hi[:, 1] - lo[:, 1])
    assert np.all(big < 0.5) and np.all(e - b < 16)
    nd = ctx.tree_nodes()
    assert len(nd["path"]) == 2 * len(b) - 1
    split = nd["ints"][:, 2] >= 0
    many = nd["ints"][:, 1] - nd["ints"][:, 0] >= 16
    assert np.array_equal(split, many | (nd["geom"][:, 2:].max(1) >= 0.5))
