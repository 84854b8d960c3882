"""Training tiles, their reduction and the weights' fragments at the sizes
where they change form: ragged tiles, fewer tiles than the waves that add them,
and the fragments an Adam step writes against those packed from its weights."""
import numpy as np
import pytest

import vvflow_amd as V
from cases import random_cluster_case, rel_l2
from test_gpu_farfield import M, sample_model
from test_gpu_parity import load_case

pytestmark = pytest.mark.gpu


@pytest.fixture(scope="module")
def ctx():
    c = V.Context(0)
    yield c
    c.close()


def data(n, seed):
    r = np.random.default_rng(seed)
    X = (r.normal(size=(n, 12)) * r.uniform(0.3, 3, 12) + r.normal(size=12)).astype(np.float32)
    Y = (r.normal(size=(n, 2)) * [0.1, 0.2]).astype(np.float32)
    return X, Y, r.uniform(0.5, 1.5, n).astype(np.float32)


@pytest.mark.parametrize("n", [1, 31, 33, 511, 512, 545, 5000])
def test_gradients_vs_oracle(ctx, n):
    print(f"case train tiles n={n}", flush=True)
    X, Y, W = data(n, n)
    p = sample_model(*data(4096, 1)[:2], seed=n)
    ctx.far_model_set(p)
    lg, gg = ctx.far_gradients(X, Y, W)
    lo, go = M.loss_and_grad(p, X, Y, W, mirror=True)
    assert np.isclose(lg, lo, rtol=1e-3)
    # bf16 operands (2^-9 each) and flips of the mirrored roundings
    for a, b in ((M.O_W1, M.O_B1), (M.O_B1, M.O_W2), (M.O_W2, M.O_B2), (M.O_B2, M.O_W3), (M.O_W3, M.O_B3),
                 (M.O_B3, M.N_TRAIN)):
        assert rel_l2(gg[a:b], go[a:b]) < 1e-2, (a, b)


@pytest.mark.parametrize("batch", [32, 544, 4096])
def test_fragments_follow_the_weights(ctx, batch):
    print(f"case fragments batch={batch}", flush=True)
    X, Y, W = data(6000, batch)
    objs = random_cluster_case(3000, batch, "cluster")
    ctx.far_model_set(sample_model(X, Y))
    ctx.far_train_data(X, Y, W)
    loss = ctx.far_train(np.full(5, 1e-2, np.float32), batch=batch, seed=2)
    assert np.all(np.isfinite(loss)) and np.all(loss > 0)
    other = V.Context(0)   # packs the trained weights anew
    try:
        other.far_model_set(ctx.far_model_get())
        assert np.array_equal(ctx.far_forward(X), other.far_forward(X))
        for a, b in zip(ctx.far_gradients(X, Y, W), other.far_gradients(X, Y, W)):
            assert np.array_equal(a, b)
        for c in (ctx, other):
            load_case(c, objs)
            c.tree_build(8)
            c.epsilon(False)
            c.convective_learned()
        # the same kernels on the same state
        assert np.allclose(ctx.download()[:, 3:5], other.download()[:, 3:5], rtol=1e-12, atol=1e-15)
    finally:
        other.close()
