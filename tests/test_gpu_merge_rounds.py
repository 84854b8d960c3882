"""The merges of epsilon (vortices and heat particles) as a fixed point of
parallel rounds against the oracle's sequential ones, bit for bit: lists whose
merges wait for each other in long chains, from one particle up."""
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


def ring(n, pitch, signs, seed):
    """n particles one after another along the wall, `pitch` segment lengths
    apart: each one's partner is its neighbour's partner too."""
    r = np.random.default_rng(seed)
    dl = 2 * 0.5 * np.sin(np.pi / 200)
    th = 0.3 + np.arange(n) * pitch * dl / 0.502
    o = np.zeros((n, 6))
    o[:, 0], o[:, 1] = 0.502 * np.cos(th), 0.502 * np.sin(th)
    o[:, 2] = r.uniform(0.5, 1.5, n) * 1e-3
    if signs == "alternating":
        o[:, 2] *= np.where(np.arange(n) % 2, -1, 1)
    elif signs == "equal and opposite":
        o[:, 2] = np.where(np.arange(n) % 2, -1e-3, 1e-3)
    return o


def cloud(n, seed):
    """A dense layer at the wall, mixed signs, some particles twice or without
    circulation: most of it merges away."""
    r = np.random.default_rng(seed)
    th, rr = r.uniform(0, 2 * np.pi, n), 0.501 + r.exponential(0.01, n)
    o = np.zeros((n, 6))
    o[:, 0], o[:, 1] = rr * np.cos(th), rr * np.sin(th)
    o[:, 2] = r.normal(size=n) * 1e-3
    o[n // 2:n // 2 + n // 50, :2] = o[:n // 50, :2]
    o[r.random(n) < 0.02, 2] = 0
    return o


def wide(n, seed):
    """Such layers strung out downstream: leaves by the ten thousand."""
    o = cloud(n, seed)
    o[:, 0] += np.floor(np.random.default_rng(seed + 1).uniform(0, 800, n)) * 1.3
    return o


KINDS = {"ring": None, "cloud": cloud, "wide": wide}
CASES = [("ring", 1, 0.1, "same"), ("ring", 2, 0.1, "same"), ("ring", 3, 0.1, "alternating"),
         ("ring", 17, 0.05, "same"), ("ring", 65, 0.2, "equal and opposite"), ("ring", 300, 0.02, "same"),
         ("ring", 700, 0.3, "alternating"), ("cloud", 500, 5, ""), ("cloud", 3000, 6, ""),
         # more targets than one workgroup applies, and more chunks of 256 leaves than a wave tests at once
         ("cloud", 30000, 7, ""), ("wide", 250000, 8, "")]


@pytest.mark.parametrize("kind,n,a,signs", CASES)
def test_merge_rounds_vs_oracle(ctx, kind, n, a, signs):
    print(f"case merge rounds {kind} n={n} {a} {signs}", flush=True)
    v = ring(n, a, signs, n) if kind == "ring" else KINDS[kind](n, a)
    h = ring(n, a, "same", n + 1) if kind == "ring" else KINDS[kind](n, a + 100)
    h[:, 2] = np.abs(h[:, 2])
    corners = cylinder_corners(200)
    dl = 200 * np.sin(np.pi / 200) / 199
    tree = (8, 5 * dl, 100 * dl)
    o = oracle_for(v, corners=corners)
    o.set_list(V.LIST_HEAT, h)
    mirror(ctx, o)
    o.tree_build(*tree)
    ctx.tree_build(*tree)
    nn1o, nn2o, _, mo = o.epsilon(True)
    nn1, nn2, mg = ctx.epsilon(True, want_nn=True)
    print(f"  merged {mg} of {2 * n}", flush=True)
    assert mg == mo
    assert np.array_equal(nn1, nn1o) and np.array_equal(nn2, nn2o)
    keep = [0, 1, 2, 5]
    assert np.array_equal(ctx.download()[:, keep], o.vortices()[:, keep])
    assert np.array_equal(ctx.download_list(V.LIST_HEAT)[:, keep], o.get_list(V.LIST_HEAT)[:, keep])
