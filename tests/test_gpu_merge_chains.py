"""Merges that wait for each other one by one, bit for bit against the oracle's
sequential ones: chains longer than the rounds wait for, whose targets are then
visited in order (more of them than one launch visits; leaves of hundreds;
several simulations side by side; heat particles)."""
import numpy as np
import pytest

import vvflow_amd as V
from cases import cylinder_corners, oracle_for
from test_gpu_heat import body_record, mirror
from test_gpu_merge_rounds import cloud, ring

pytestmark = pytest.mark.gpu

DL = 200 * np.sin(np.pi / 200) / 199
KEEP = [0, 1, 2, 5]


@pytest.fixture(scope="module")
def ctx():
    c = V.Context(0)
    yield c
    c.close()


def line(n, pitch, x0=1.0):
    """n equal particles in a row: each one's merge decides the next one's."""
    o = np.zeros((n, 6))
    o[:, 0] = x0 + np.arange(n) * pitch
    o[:, 2] = 1e-3
    return o


def lines(n, rows):
    return np.concatenate([line(n, 1e-4, 1.0 + 0.01 * k) + [0, 0.05 * k, 0, 0, 0, 0] for k in range(rows)])


LISTS = {"line 40": lambda: line(40, 1e-3), "line 2000": lambda: line(2000, 1e-4), "line 5001": lambda: line(5001, 5e-5),
         "spread line": lambda: line(3000, 2e-3), "rows": lambda: lines(700, 6), "ring": lambda: ring(1500, 0.02, "same", 3),
         "ring and cloud": lambda: np.concatenate([ring(900, 0.02, "same", 4), cloud(2000, 9) + [3, 0, 0, 0, 0, 0]]),
         "cancelling": lambda: ring(1200, 0.02, "equal and opposite", 5)}


@pytest.mark.parametrize("least", [0.0, 5 * DL])   # leaves of a few, or of what a length of 5 DL holds
@pytest.mark.parametrize("name", list(LISTS))
def test_chains_vs_oracle(ctx, name, least):
    print(f"case merge chain {name} least node {least:.3f}", flush=True)
    v = LISTS[name]()
    h = v.copy()
    h[:, 2] = np.abs(h[:, 2])
    o = oracle_for(v, corners=cylinder_corners(200))
    o.set_list(V.LIST_HEAT, h)
    mirror(ctx, o)
    o.tree_build(8, least, 100 * DL)
    ctx.tree_build(8, least, 100 * DL)
    nn1o, nn2o, _, mo = o.epsilon(True)
    nn1, nn2, mg = ctx.epsilon(True, want_nn=True)
    print(f"  merged {mg} of {2 * len(v)}", flush=True)
    assert mg == mo
    assert np.array_equal(nn1, nn1o) and np.array_equal(nn2, nn2o)
    assert np.array_equal(ctx.download()[:, KEEP], o.vortices()[:, KEEP])
    assert np.array_equal(ctx.download_list(V.LIST_HEAT)[:, KEEP], o.get_list(V.LIST_HEAT)[:, KEEP])


@pytest.mark.parametrize("names", [("line 40", "line 2000"), ("ring", "line 5001", "ring and cloud", "line 40", "rows")])
def test_chains_of_a_batch(ctx, names):
    print(f"case merge chains batch {names}", flush=True)
    parts = [LISTS[k]() for k in names]
    off = np.concatenate([[0], np.cumsum([len(p) for p in parts])])
    segs, body, ref, merged = [], [], [], 0
    for k, p in enumerate(parts):
        o = oracle_for(p, corners=cylinder_corners(200))
        segs.append(np.ascontiguousarray(o.segments(), dtype=V.SEG_DTYPE))
        body.append(body_record(o))
        body[-1]["first_seg"] = 200 * k
        o.tree_build(8, 5 * DL, 100 * DL)
        merged += o.epsilon(True)[3]
        ref.append(o.vortices())
    ctx.set_params(re=600.0, dt=0.005)
    for kind in (V.LIST_HEAT, V.LIST_STREAK):
        ctx.upload_list(kind, np.zeros((0, 6)))
    ctx.upload_bodies(np.concatenate(segs), np.concatenate(body))
    ctx.upload(np.concatenate(parts))
    ctx.set_batch(off, np.arange(len(parts) + 1), [600.0] * len(parts))
    ctx.tree_build(8, 5 * DL, 100 * DL)
    assert ctx.epsilon(True) == merged
    assert np.array_equal(ctx.download()[:, KEEP], np.concatenate(ref)[:, KEEP])
