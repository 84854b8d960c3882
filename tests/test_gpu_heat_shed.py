"""Shedding of heat by every condition against the oracle, bit for bit: fewer
and more segments than a block has threads, layer particles used once, by
several segments, and not yet there."""
import numpy as np
import pytest

import vvflow_amd as V
from cases import cylinder_corners, oracle_for
from test_gpu_heat import HEAT, mirror

pytestmark = pytest.mark.gpu


@pytest.fixture(scope="module")
def ctx():
    c = V.Context(0)
    yield c
    c.close()


CASES = [(cond, nseg, layer) for cond in (V.HC_ISOLATE, V.HC_CONST_T, V.HC_CONST_W) for nseg in (3, 64, 1023, 1025, 2600)
         for layer in ("none",)] + [(V.HC_CONST_T, nseg, layer) for nseg in (3, 64, 1025)
                                    for layer in ("once", "shared", "new")]


@pytest.mark.parametrize("cond,nseg,layer", CASES)
def test_heat_shed_vs_oracle(ctx, cond, nseg, layer):
    print(f"case heat shed {cond} nseg={nseg} {layer}", flush=True)
    r = np.random.default_rng(nseg)
    nh = 50
    h = np.zeros((nh, 6))
    h[:, :2] = r.uniform(1, 2, (nh, 2))
    h[:, 2] = r.uniform(0.5, 2, nh) * 1e-3
    o = oracle_for(np.zeros((0, 6)), corners=cylinder_corners(nseg))
    segs = o.segments()
    segs["hsum"] = r.normal(size=nseg) * (r.random(nseg) < 0.7)
    o.set_segments(segs)
    hc = r.uniform(0.5, 1.5, nseg).astype(np.float32)
    o.set_heat([cond], hc)
    o.set_list(HEAT, h)
    lay = np.full(nseg, -1, dtype=np.int64)
    if layer == "once":
        k = min(nseg, nh)
        lay[r.permutation(nseg)[:k // 2 + 1]] = r.permutation(nh)[:k // 2 + 1]
    elif layer == "shared":
        lay[::2] = r.integers(0, 5, len(lay[::2]))
    elif layer == "new":
        lay[-1] = nh   # the particle that the first segment sheds
    mirror(ctx, o)
    ctx.set_heat([cond], hc)
    o.set_heat_layer(lay)
    ctx.set_heat_layer(lay)
    o.heat_shed()
    ctx.heat_shed()
    assert np.array_equal(ctx.download_list(HEAT), o.get_list(HEAT))
    assert np.array_equal(ctx.download_bodies()[0]["hsum"], o.segments()["hsum"])
