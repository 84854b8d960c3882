"""Near and far lists against the oracle's, entry for entry: groups of leaves
of every remainder, walks cut into several items, far criteria from none near
to all near (the logs then run out of the room they start with)."""
import numpy as np
import pytest

import vvflow_amd as V
from cases import oracle_for, path_code32, random_cluster_case
from test_gpu_parity import load_case

pytestmark = pytest.mark.gpu

CASES = [(1, 8), (17, 8), (900, 0), (900, 8), (1100, 300), (20000, 0), (20000, 8), (20000, 1000),
         (20000, 10**9), (65000, 10**9)]


@pytest.mark.parametrize("n,fc", CASES)
def test_lists_vs_oracle(n, fc):
    print(f"case lists n={n} fc={fc}", flush=True)
    objs = random_cluster_case(n, n + 1)
    o = oracle_for(objs)
    o.tree_build(fc)
    t = o.tree()
    depth = np.zeros(len(t["path"]), dtype=np.int64)
    for i in range(1, len(depth)):
        depth[i] = depth[t["ints"][i, 3]] + 1
    code = path_code32(t["path"])
    ctx = V.Context(0)   # new logs
    try:
        load_case(ctx, objs)
        for _ in range(2):   # the second walk has the grown logs
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
