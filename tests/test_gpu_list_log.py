"""The log of the list builder where one group of leaves needs far more room
than the others: strays spread wide around a wake share a leaf that is near to
all of it.  Lists against the oracle's, entry for entry, and the device memory
that the strays cost."""
import numpy as np
import pytest
import torch

import vvflow_amd as V
from cases import oracle_for, path_code32, random_cluster_case
from test_gpu_parity import load_case

pytestmark = pytest.mark.gpu


def with_strays(n, k, seed):
    r = np.random.default_rng(seed)
    o = random_cluster_case(n + k, seed)
    o[n:, 0], o[n:, 1] = r.uniform(-200, -10, k), r.uniform(-100, 100, k)
    return o


# a walk of 65000 has about 110 items, room for 64 is kept from the start
@pytest.mark.parametrize("n,k,fc", [(65000, 10, 8), (65000, 10, 1000), (65000, 40, 8), (3000, 10, 8)])
def test_lists_with_strays_vs_oracle(n, k, fc):
    print(f"case list log n={n} strays={k} fc={fc}", flush=True)
    objs = with_strays(n, k, n + k)
    o = oracle_for(objs)
    o.tree_build(fc)
    t = o.tree()
    depth = np.zeros(len(t["path"]), dtype=np.int64)
    for i in range(1, len(depth)):
        depth[i] = depth[t["ints"][i, 3]] + 1
    code = path_code32(t["path"])
    ctx = V.Context(0)
    try:
        # room from the start, as the walk before needed it, and as one of
        # another criterion needed it
        for before in (None, fc, 10**9 if n < 10000 else 0):
            load_case(ctx, objs)
            if before is not None:
                ctx.tree_build(before)
                ctx.tree_destroy()
                load_case(ctx, objs)
            ctx.tree_build(fc)
            for far in (False, True):
                g = ctx.tree_lists(far=far)
                off, nodes = t["far" if far else "near"]
                assert np.array_equal(g["off"], off)
                assert np.array_equal(path_code32(g["path"]), code[nodes])
                assert np.array_equal(g["depth"], depth[nodes])
            ctx.tree_destroy()
    finally:
        ctx.close()


def test_memory_of_strays():
    """Ten strays lengthen the lists by one wide leaf's; the room of the other
    16000 leaves stays as it is without them."""
    used = []
    for k in (0, 10):
        print(f"case list log memory strays={k}", flush=True)
        objs = np.concatenate([V.gen_wake(1000000), with_strays(0, k, 5)])
        ctx = V.Context(0)
        try:
            ctx.upload(objs)
            torch.cuda.synchronize()
            free = torch.cuda.mem_get_info()[0]
            ctx.tree_build(8)
            torch.cuda.synchronize()
            used.append((free - torch.cuda.mem_get_info()[0]) / 2**20)
        finally:
            ctx.close()
    print(f"  {used[0]:.0f} and {used[1]:.0f} MiB", flush=True)
    assert used[1] < 1.25 * used[0]


def test_little_memory_left():
    """A tree of 2.2M vortices with 2.9 GiB of device memory left: its lists are
    walked in parts, and are those that a walk of all has."""
    n = 2200000
    objs = V.gen_wake(n)
    out = []
    for left in (None, 2.9):
        print(f"case list log n={n}, GiB left: {left}", flush=True)
        ctx = V.Context(0)
        hog = None
        try:
            ctx.upload(objs)
            ctx.snapshot()
            torch.cuda.synchronize()
            if left:
                torch.cuda.empty_cache()
                hog = torch.empty(torch.cuda.mem_get_info()[0] - int(left * 2**30), dtype=torch.uint8, device="cuda")
            for _ in range(2):   # without and with the buffers of the build before
                ctx.restore()
                ctx.tree_build(8)
            hog = None
            torch.cuda.empty_cache()
            near = ctx.tree_lists()
            ctx.epsilon(False)
            ctx.convective((1.0, 0.0))
            out.append((near["off"], near["path"], near["depth"], ctx.download()))
            ctx.restore()
            ctx.tree_build(8)   # memory again
            ctx.epsilon(False)
            ctx.convective((1.0, 0.0))
            assert np.array_equal(ctx.download(), out[0][3])
        finally:
            ctx.close()
    for a, b in zip(*out):
        assert np.array_equal(a, b)
