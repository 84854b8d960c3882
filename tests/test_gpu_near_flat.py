"""Sums over a leaf list as one sequence of elements, against the oracle:
velocities at few points (sources read in place) and many (packed sources), and
leaves of more elements than the table of a wave holds at once."""
import numpy as np
import pytest

import vvflow_amd as V
from cases import oracle_for, random_cluster_case
from test_gpu_parity import load_case

pytestmark = pytest.mark.gpu


@pytest.fixture(scope="module")
def ctx():
    c = V.Context(0)
    yield c
    c.close()


# packed from 256 points on; a leaf of at least min_node holds
# all its elements (min_node 2 and more: the root alone)
@pytest.mark.parametrize("n,npts,min_node", [(1, 1, 0.0), (1000, 255, 0.0), (1000, 256, 0.0), (1000, 400, 0.0),
                                             (1024, 5, 2.0), (1025, 40, 2.0), (3000, 5, 2.0), (3000, 300, 0.4)])
def test_point_sums_vs_oracle(ctx, n, npts, min_node):
    print(f"case near flat n={n} npts={npts} min={min_node}", flush=True)
    objs = random_cluster_case(n, n + npts)
    o = oracle_for(objs)
    load_case(ctx, objs)
    o.tree_build(8, min_node)
    ctx.tree_build(8, min_node)
    o.epsilon(False)
    ctx.epsilon(False)
    r = np.random.default_rng(npts)
    pts = r.uniform(-0.2, 1.2, (npts, 2))
    pts[:npts // 2] = objs[r.integers(0, n, npts // 2), :2]   # on vortices
    ref, got = o.velocity(pts), ctx.velocity(pts, inf=(1.0, 0.0))
    # a term is at most |g| / (2 eps) / (2 pi) and off by under 8 roundings; n
    # of them added in two orders
    v = o.vortices()
    bound = 2 * (n + 8) * 2.0**-53 * (1 + np.sum(np.abs(v[:, 2]) * v[:, 5]) / (4 * np.pi))
    assert np.abs(got - ref).max() < bound
    assert np.array_equal(ctx.eps2h(pts), o.eps2h(pts))
