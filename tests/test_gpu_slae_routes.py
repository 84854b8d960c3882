"""The ways a boundary system is solved: with its factors when its segment rows
are new, with their inverse when they are seen again, for one system and for a
batch, and for bodies that change at every call."""
import numpy as np
import pytest

import vvflow_amd as V
from test_gpu_slae_core import scene, solution

pytestmark = pytest.mark.gpu


@pytest.fixture(scope="module")
def ctx():
    c = V.Context(0)
    yield c
    c.close()


def call(ctx, parts, time, height):
    """One calc_circulation of the parts as a batch, their bodies and vortices
    squeezed to `height`; every system and its solution."""
    segs = np.concatenate([p[0] for p in parts])
    bodies = np.concatenate([p[1] for p in parts])
    bodies["first_seg"] = np.concatenate([[0], np.cumsum(bodies["nseg"])[:-1]])
    for f in ("cy", "y", "dly"):
        segs[f] *= height
    v = np.concatenate([p[2] for p in parts])
    v[:, 1] *= height
    ctx.set_params(re=600.0, dt=0.005, time=time)
    ctx.upload_bodies(segs, bodies)
    ctx.upload(v)
    if len(parts) > 1:
        ctx.set_batch([400 * k for k in range(len(parts) + 1)],
                      np.concatenate([[0], np.cumsum([len(p[1]) for p in parts])]), [600.0] * len(parts))
    ctx.tree_build(8, 0.05, 10.0)
    ctx.epsilon(False)
    ctx.calc_circulation((1.0, 0.2))
    s, b = ctx.download_bodies()
    out, k = [], 0
    for p in parts:
        out.append(solution(s, b[k:k + len(p[1])]))
        k += len(p[1])
    return out


CASES = [((41,),), ((129,),), ((20, 7, 50),), ((41,), (16, 16)), ((33,), (33,), (33,))]


@pytest.mark.parametrize("sizes", CASES)
def test_factors_and_inverse(ctx, sizes):
    print(f"case slae routes {sizes}", flush=True)
    parts = [scene(z, 3 + k, shift=5.0 * k) for k, z in enumerate(sizes)]
    # heights of successive calls: new, seen again (inverse made), again, changed
    # every call, seen again, and at time 0 always new
    got = {}
    for time, h in ((0.5, 1.0), (0.5, 1.0), (0.5, 1.0), (0.5, 0.7), (0.5, 0.5), (0.5, 1.0), (0.5, 0.7), (0.5, 0.7),
                    (0.0, 0.7), (0.0, 0.7), (0.5, 0.7)):
        got.setdefault(h, []).append(call(ctx, parts, time, h))
    for h, calls in got.items():
        call(ctx, parts[:1], 0.0, h)
        A, b = ctx.slae_system()
        ref = np.linalg.solve(A, b)
        cond = np.linalg.cond(A / np.abs(A).max(1)[:, None])
        for x in calls:
            # backward stable each: within cond * eps of the exact solution
            assert np.linalg.norm(x[0] - ref) <= 50 * cond * 2.3e-16 * np.linalg.norm(ref)
            for k in range(len(parts)):
                assert np.linalg.norm(x[k] - calls[0][k]) <= 100 * cond * 2.3e-16 * np.linalg.norm(calls[0][k])
