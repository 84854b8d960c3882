"""Flow-move of heat and streak lists of more particles than waves that take one
each, bit for bit against the oracle: lists at and round the size from which a
wave takes two and more, near a star body and without one."""
import numpy as np
import pytest

import vvflow_amd as V
from cases import oracle_for
from test_gpu_heat import HEAT, STREAK, mirror

pytestmark = pytest.mark.gpu


@pytest.fixture(scope="module")
def ctx():
    c = V.Context(0)
    yield c
    c.close()


def star():
    k = np.arange(24)
    rad, ang = np.where(k % 2 == 0, 1.0, 0.55), 2 * np.pi - np.pi * k / 12
    return np.stack([rad * np.cos(ang), rad * np.sin(ang)], 1)


# a wave takes two from 131072 particles on
@pytest.mark.parametrize("nh,ns,body", [(131071, 63, True), (131072, 131073, True), (200003, 1, True), (1, 1, False),
                                        (63, 65, False), (1000, 131072, False)])
def test_many_particles_vs_oracle(ctx, nh, ns, body):
    print(f"case passive move heat={nh} streak={ns} body={body}", flush=True)
    r = np.random.default_rng(nh + ns)
    lists = []
    for n in (nh, ns):
        a = np.zeros((n, 6))
        a[:, :2] = r.uniform(-1.5, 1.5, (n, 2))
        a[:, 2] = r.uniform(0.5, 2, n) * 1e-3
        a[::37, 2] = 3e-11   # below remove_eps
        a[:, 3:5] = r.normal(size=(n, 2)) * 0.2
        lists.append(a)
    o = oracle_for(np.zeros((0, 6)), corners=star() if body else None, dt=0.01)
    hc = r.uniform(0.5, 1.5, 24).astype(np.float32)
    if body:
        o.set_heat([V.HC_CONST_T], hc)
    o.set_list(HEAT, lists[0])
    o.set_list(STREAK, lists[1])
    mirror(ctx, o, dt=0.01)
    if body:
        ctx.set_heat([V.HC_CONST_T], hc)
    for step in range(2):
        o.move_and_clean(True)
        ctx.move_and_clean(True)
        for lid in (HEAT, STREAK):
            assert np.array_equal(ctx.download_list(lid), o.get_list(lid))
        if body:
            assert np.array_equal(ctx.heat_layer(), o.heat_layer())
            assert np.array_equal(ctx.download_bodies()[0]["hsum"], o.segments()["hsum"])
        # the lists lie still after the first move: another one of their own
        for lid in (HEAT, STREAK):
            a = o.get_list(lid)
            a[:, 3:5] = r.normal(size=(len(a), 2)) * 0.2
            o.set_list(lid, a)
            ctx.upload_list(lid, a)
        if body:
            ctx.set_heat_layer(o.heat_layer())
