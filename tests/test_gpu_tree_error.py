"""Tree builds that end in an error: the list keeps its records, and no call
takes what is there for a tree."""
import numpy as np
import pytest
import torch

import vvflow_amd as V
from cases import random_cluster_case
from test_gpu_heat import HEAT, STREAK

pytestmark = pytest.mark.gpu

def rows(a):
    return a[np.lexsort(a.T)]


def refused(ctx):
    for call in (lambda: ctx.convective((1.0, 0.0)), lambda: ctx.epsilon(True), ctx.diffusive, ctx.tree_leaves,
                 lambda: ctx.velocity(np.zeros((1, 2)))):
        with pytest.raises(V.VVHDError, match="tree is not built"):
            call()


@pytest.mark.parametrize("n", [12, 1600, 40000])
@pytest.mark.parametrize("built", [False, True])
def test_a_tree_without_an_end(n, built):
    """Least and largest node sizes under which a single element splits for
    ever: refused, with or without a tree of before."""
    print(f"case tree error n={n} built before: {built}", flush=True)
    v = random_cluster_case(n, n)
    v[:, 3:6] = np.random.default_rng(n).normal(size=(n, 3))
    h = random_cluster_case(30, 1)
    h[:, 3] = np.arange(30)
    ctx = V.Context(0)
    try:
        ctx.upload(v)
        ctx.upload_list(HEAT, h)
        ctx.upload_list(STREAK, h[:7])
        if built:
            ctx.tree_build(8)
        with pytest.raises(V.VVHDError, match="tree_build"):
            ctx.tree_build(8, -1.0, 0.0)
        refused(ctx)
        assert np.array_equal(rows(ctx.download()), rows(v))
        assert np.array_equal(rows(ctx.download_list(HEAT)), rows(h))
        assert np.array_equal(rows(ctx.download_list(STREAK)), rows(h[:7]))
        ctx.tree_build(8)
        ctx.epsilon(False)
    finally:
        ctx.close()


def test_a_tree_without_memory():
    n = 2200000
    print(f"case tree error n={n} without memory", flush=True)
    v = V.gen_wake(n)
    ctx = V.Context(0)
    try:
        ctx.upload(v)
        torch.cuda.synchronize()
        torch.cuda.empty_cache()
        hog = torch.empty(torch.cuda.mem_get_info()[0] - (1 << 30), dtype=torch.uint8, device="cuda")
        with pytest.raises(V.VVHDError, match="hipMalloc"):
            ctx.tree_build(8)
        refused(ctx)
        del hog
        torch.cuda.empty_cache()
        assert np.array_equal(rows(ctx.download()), rows(v))
        ctx.tree_build(8)
        ctx.epsilon(False)
        ctx.convective((1.0, 0.0))
    finally:
        ctx.close()
