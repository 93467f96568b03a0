"""The outputs a loss is taken of are those of the last prediction, whatever happened to the network since and
wherever the prediction went: into a shared FP32 batch (written there by the product itself) or by way of rows
(FP64 batches).  Both give the same loss and gradients, to the bit: the outputs are the same sums through the
same map, and everything behind them is one code."""
import numpy as np
import pytest

from spock_amd import runtime as rt

pytestmark = pytest.mark.gpu


@pytest.fixture(scope="module")
def ctx():
    return rt.Context(0)


def nothing(mlp, batch, x0):
    pass


def parameters(mlp, batch, x0):
    mlp.set_params(-2.0 * mlp.params())


def normalization(mlp, batch, x0):
    a, b, c, d = mlp.normalization()
    mlp.set_normalization(a, b, c + 1.0, 3.0 * d)


def adam(mlp, batch, x0):
    mlp.adam(lr=0.1)
    mlp.adam(lr=0.1)


def dataset(mlp, batch, x0):
    mlp.dataset(batch, x0)


@pytest.mark.parametrize("change", [nothing, parameters, normalization, adam, dataset], ids=lambda f: f.__name__)
@pytest.mark.parametrize("layers", [0, 2])
def test_loss_of_the_last_prediction(ctx, problem_dirs, change, layers):
    p = rt.Problem(ctx, problem_dirs["small"])
    n, nx, count = p.n_iter, p.nx, 40
    rng = np.random.default_rng(11)
    x0 = rng.standard_normal((count, nx))
    target = rng.standard_normal((count, n)).astype(np.float32)
    start = rng.standard_normal((count, n))
    shift, scale = rng.standard_normal(n), 0.1 + rng.random(n)
    found = []
    for dtype in (rt.F64, rt.F32):
        mlp = rt.WarmStartMLP(ctx, nx, n, hidden=24, layers=layers, seed=5)
        mlp.set_normalization(np.zeros(nx), np.full(nx, 0.5), shift, scale)
        mlp.forward(x0.astype(np.float32))
        mlp.loss_backward(target)  # gradients for Adam
        data = rt.Batch(ctx, [p] * count, rt.F64, shared=True)
        data.set_iterates(start)
        mlp.predict(x0, rt.Batch(ctx, [p] * count, dtype, shared=True))
        change(mlp, data, x0)
        loss = mlp.loss_backward(target)
        found.append((loss, mlp.grads()))
    assert np.isfinite(found[0][0])
    assert found[0][0] == found[1][0]
    assert np.array_equal(found[0][1], found[1][1])
