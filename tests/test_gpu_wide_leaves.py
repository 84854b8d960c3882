"""Sums over near leaves of very unequal sizes against the oracle: leaves that a
lane writes into the wave's table, that all lanes write, and that are read
without it, alone and side by side; ordered (friction, boundary system) and not."""
import numpy as np
import pytest

import vvflow_amd as V
from cases import cylinder_corners, oracle_for
from test_gpu_heat import mirror

pytestmark = pytest.mark.gpu


@pytest.fixture(scope="module")
def ctx():
    c = V.Context(0)
    yield c
    c.close()


def lumps(sizes, seed):
    """Clusters of the given sizes on a circle round a body, each smaller than
    the least node size and so a leaf (with what is left of its neighbours)."""
    r = np.random.default_rng(seed)
    o = np.zeros((sum(sizes), 6))
    at = np.repeat(np.arange(len(sizes)), sizes)
    th = 2 * np.pi * at / len(sizes)
    o[:, 0] = 0.8 * np.cos(th) + r.uniform(-0.02, 0.02, len(at))
    o[:, 1] = 0.8 * np.sin(th) + r.uniform(-0.02, 0.02, len(at))
    o[:, 2] = r.choice([-1.0, 1.0], len(at)) * r.uniform(0.5, 1.5, len(at)) * 1e-3
    return o


# 32: what a lane writes by itself; 512: what goes through the table; 1024: the table
CASES = [(32,), (33,), (64, 31), (65, 32, 33), (512, 5), (513, 5), (1023, 1), (1025, 600, 2), (3, 700, 40, 1500, 16, 33, 511)]


@pytest.mark.parametrize("sizes", CASES)
def test_sums_over_unequal_leaves(ctx, sizes):
    print(f"case wide leaves {sizes}", flush=True)
    objs = lumps(sizes, len(sizes))
    n = len(objs)
    o = oracle_for(objs, corners=cylinder_corners(40))
    o.set_list(V.LIST_HEAT, np.abs(lumps(sizes, 99)) * [1, 1, 1, 0, 0, 0])
    mirror(ctx, o)
    o.tree_build(8, 0.1, 10.0)
    ctx.tree_build(8, 0.1, 10.0)
    o.epsilon(False)
    ctx.epsilon(False)
    r = np.random.default_rng(5)
    for npts in (7, 300):   # sources in place and, where leaves average up to 128, packed
        pts = r.uniform(-1, 1, (npts, 2))
        pts[::3] = objs[r.integers(0, n, len(pts[::3])), :2]
        ref, got = o.velocity(pts), ctx.velocity(pts, inf=(1.0, 0.0))
        # a term is at most |g| / (2 eps) / (2 pi) and off by under 8 roundings;
        # n of them added in two orders
        v = o.vortices()
        bound = 2 * (n + 8) * 2.0**-53 * (1 + np.sum(np.abs(v[:, 2]) * v[:, 5]) / (4 * np.pi))
        assert np.abs(got - ref).max() < bound
        assert np.array_equal(ctx.eps2h(pts), o.eps2h(pts))
    _, b_o = o.calc_circulation(want_matrix=True)
    ctx.calc_circulation((1.0, 0.0))
    _, b_g = ctx.slae_system()
    # the same additions in the same order; terms off by the library's log and
    # division, a few roundings of each
    assert np.abs(b_g - b_o).max() <= 1e-13 * max(np.abs(b_o).max(), 1.0)
    o.diffusive()
    ctx.diffusive()
    fo, fg = o.segments()["fric"], ctx.download_bodies()[0]["fric"]
    assert np.allclose(fg, fo, rtol=1e-10, atol=1e-13 * max(np.abs(fo).max(), 1e-300))
    o.diffusive_heat()
    ctx.diffusive_heat()
    ho, hg = o.get_list(V.LIST_HEAT)[:, 3:5], ctx.download_list(V.LIST_HEAT)[:, 3:5]
    assert np.linalg.norm(hg - ho) <= 1e-10 * np.linalg.norm(ho)
