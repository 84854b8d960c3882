"""calc_circulation through the core of each system (segment rows, kept
inverse) against a dense FP64 solve of the whole system that the library
filled: core sizes round the tiles, several bodies, and a batch whose systems
have one order but different numbers of bodies."""
import numpy as np
import pytest

import vvflow_amd as V

pytestmark = pytest.mark.gpu


@pytest.fixture(scope="module")
def ctx():
    c = V.Context(0)
    yield c
    c.close()


def scene(sizes, seed, shift=0.0):
    """Circles of the given segment counts side by side and vortices round
    them: segment and body records, vortex list."""
    r = np.random.default_rng(seed)
    segs, bodies = [], np.zeros(len(sizes), dtype=V.BODY_DTYPE)
    first = 0
    for b, k in enumerate(sizes):
        s = V.segments_from_corners(V.gen_cylinder(0.4, k) + [shift + 1.3 * b, 0.0])
        segs.append(s)
        bodies[b]["first_seg"], bodies[b]["nseg"] = first, k
        bodies[b]["friction_prev"] = (1e-4, -2e-4, 3e-5)
        bodies[b]["fdt_dead"] = (1e-5, 2e-5, -3e-5)
        first += k
    n = 400
    v = np.zeros((n, 6))
    v[:, 0] = r.uniform(shift - 1, shift + 1.3 * len(sizes), n)
    v[:, 1] = np.where(r.random(n) < 0.5, 1, -1) * r.uniform(0.5, 1.0, n)
    v[:, 2] = r.normal(size=n) * 1e-3
    return np.ascontiguousarray(np.concatenate(segs), dtype=V.SEG_DTYPE), bodies, v


def solution(segs, bodies):
    x = []
    for b in bodies:
        x += [segs["g"][b["first_seg"]:b["first_seg"] + b["nseg"]], b["speed_slae"], b["force_hydro"], b["force_holder"]]
    return np.concatenate(x)


@pytest.mark.parametrize("sizes", [(5,), (31,), (33,), (64,), (129,), (40, 25), (20, 7, 50)])
def test_core_solve_vs_dense(ctx, sizes):
    print(f"case slae core {sizes}", flush=True)
    segs, bodies, v = scene(sizes, sum(sizes))
    for time in (0.0, 0.5, 0.5):   # inverted, kept, kept
        ctx.set_params(re=600.0, dt=0.005, time=time)
        ctx.upload_bodies(segs, bodies)
        ctx.upload(v)
        ctx.tree_build(8, 0.05, 10.0)
        ctx.epsilon(False)
        ctx.calc_circulation((1.0, 0.2))
        A, b = ctx.slae_system()
        x = solution(*ctx.download_bodies())
        # both are backward stable: each within cond * eps of the exact solution
        ref = np.linalg.solve(A, b)
        cond = np.linalg.cond(A / np.abs(A).max(1)[:, None])
        assert np.linalg.norm(x - ref) <= 50 * cond * 2.3e-16 * np.linalg.norm(ref)
        assert np.abs(A @ x - b).max() <= 1e-11 * (np.abs(A) @ np.abs(x) + np.abs(b)).max()
        sp = ctx.download_bodies()[1]["speed_slae"]
        assert np.all(sp == 0)


def test_batch_of_unlike_bodies(ctx):
    """Systems of 9 + 41 and 2 x 9 + 32 equations in one batch: each equals
    its own run alone."""
    print("case slae core batch (41), (16, 16)", flush=True)
    parts = [scene((41,), 1), scene((16, 16), 2, shift=5.0)]
    alone = []
    for segs, bodies, v in parts:
        ctx.set_params(re=600.0, dt=0.005, time=0.0)
        ctx.upload_bodies(segs, bodies)
        ctx.upload(v)
        ctx.tree_build(8, 0.05, 10.0)
        ctx.epsilon(False)
        ctx.calc_circulation((1.0, 0.2))
        alone.append(solution(*ctx.download_bodies()))
    segs = np.concatenate([p[0] for p in parts])
    bodies = np.concatenate([p[1] for p in parts])
    bodies["first_seg"] = [0, 41, 57]
    ctx.upload_bodies(segs, bodies)
    ctx.upload(np.concatenate([p[2] for p in parts]))
    ctx.set_batch([0, 400, 800], [0, 1, 3], [600.0, 600.0])
    ctx.tree_build(8, 0.05, 10.0)
    ctx.epsilon(False)
    ctx.calc_circulation((1.0, 0.2))
    s, b = ctx.download_bodies()
    b = b.copy()
    got = [solution(s[:41], b[:1])]
    b["first_seg"] -= 41
    got.append(solution(s[41:], b[1:]))
    for g, a in zip(got, alone):
        assert np.linalg.norm(g - a) <= 1e-11 * np.linalg.norm(a)
