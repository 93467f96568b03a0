"""The network's matrix products at the edges of their tiles: operands narrower than one vector (fewer
than 4 rows), odd widths (vectors that start anywhere), one more or less than a tile of 32, 64 and 128 or a
k-step of 64 and 256, products small and large enough for either kernel, split and whole sums, and the
training step that updates a layer in the epilogue of its gradient.

The model is float64 with the kernels' inputs rounded to bfloat16.  Bounds are propagated in absolute
values: a bfloat16 rounding of an intermediate (activation, output gradient) moves it by 2^-8 of itself at
most (unit roundoff 2^-9, and a rounding that goes the other way because the FP32 sum differs), FP32 sums of
K products by K 2^-22 of the sum of magnitudes, GELU and its derivative by 2^-20."""
import numpy as np
import pytest
from scipy.special import erf

from spock_amd import runtime as rt

pytestmark = pytest.mark.gpu


@pytest.fixture(scope="module")
def ctx():
    return rt.Context(0)


def bf16(a):
    u = np.ascontiguousarray(a, dtype=np.float32).view(np.uint32).astype(np.uint64)
    u = ((u + 0x7FFF + ((u >> 16) & 1)) >> 16) << 16
    return (u & 0xFFFFFFFF).astype(np.uint32).view(np.float32).astype(np.float64)


def gelu(x):
    return 0.5 * x * (1.0 + erf(x / np.sqrt(2.0)))


def gelu_grad(x):
    return 0.5 * (1.0 + erf(x / np.sqrt(2.0))) + x * np.exp(-0.5 * x * x) / np.sqrt(2.0 * np.pi)


SIZES = [  # in, hidden, out, rows
    (1, 1, 1, 1), (2, 3, 2, 3), (3, 5, 7, 33), (50, 63, 127, 31), (50, 65, 129, 32), (7, 256, 257, 63),
    (31, 255, 64, 65), (33, 320, 8192, 64), (5, 33, 33001, 130), (13, 129, 11001, 385),
]


@pytest.mark.parametrize("n_in,hidden,n_out,rows", SIZES)
def test_products_at_tile_edges(ctx, n_in, hidden, n_out, rows):
    mlp = rt.WarmStartMLP(ctx, n_in, n_out, hidden=hidden, layers=1, seed=3)
    rng = np.random.default_rng(n_in + hidden + n_out + rows)
    p = (rng.standard_normal(mlp.n_params) * 0.1).astype(np.float32)
    mlp.set_params(p)
    x = rng.standard_normal((rows, n_in)).astype(np.float32)
    t = rng.standard_normal((rows, n_out)).astype(np.float32)
    y = mlp.forward(x)
    loss = mlp.loss_backward(t)
    g = mlp.grads()

    e, s = 2.0 ** -8, 2.0 ** -22
    o1, o2, o3 = n_in * hidden, n_in * hidden + hidden, n_in * hidden + hidden + hidden * n_out
    p64 = p.astype(np.float64)
    X, W0, b0 = bf16(x), bf16(p[:o1]).reshape(n_in, hidden), p64[o1:o2]
    W1, b1 = bf16(p[o2:o3]).reshape(hidden, n_out), p64[o3:]
    z = X @ W0 + b0
    dz = (n_in + 1) * s * (np.abs(X) @ np.abs(W0) + np.abs(b0))
    a = gelu(z)
    da = 1.13 * dz + e * np.abs(a) + 2.0 ** -20
    ref = a @ W1 + b1
    mag = np.abs(a) @ np.abs(W1) + np.abs(b1)
    dref = da @ np.abs(W1) + (hidden + 1) * s * mag
    assert np.all(np.abs(y - ref) <= dref)
    n = rows * n_out
    dY = 2.0 * (ref - t) / n
    ddY = 2.0 * dref / n + e * np.abs(dY)
    assert abs(loss - np.mean((ref - t) ** 2)) <= np.mean(2 * np.abs(ref - t) * dref + dref ** 2) + 1e-12
    gW1, gb1 = a.T @ dY, dY.sum(0)
    bW1 = (np.abs(a) + da).T @ (np.abs(dY) + ddY) * (1 + rows * s) - np.abs(a).T @ np.abs(dY)
    assert np.all(np.abs(g[o2:o3].reshape(hidden, n_out) - gW1) <= bW1 + 1e-30)
    assert np.all(np.abs(g[o3:] - gb1) <= (ddY.sum(0) + rows * s * np.abs(dY).sum(0)))
    back = dY @ W1.T
    dback = ddY @ np.abs(W1).T + n_out * s * (np.abs(dY) @ np.abs(W1).T)
    dZ = back * gelu_grad(z)
    ddZ = 1.13 * dback + (np.abs(back) + dback) * (2 * dz + 2.0 ** -20) + e * np.abs(dZ)
    gW0, gb0 = X.T @ dZ, dZ.sum(0)
    bW0 = np.abs(X).T @ ddZ + rows * s * (np.abs(X).T @ (np.abs(dZ) + ddZ))
    assert np.all(np.abs(g[:o1].reshape(n_in, hidden) - gW0) <= bW0 + 1e-30)
    assert np.all(np.abs(g[o1:o2] - gb0) <= ddZ.sum(0) + rows * s * np.abs(dZ).sum(0) + 1e-30)


@pytest.mark.parametrize("problem", ["small", "mid"])
@pytest.mark.parametrize("hidden,layers,count", [(1, 1, 17), (65, 2, 40), (64, 0, 33)])
def test_predictions_and_training_step(ctx, problem_dirs, problem, hidden, layers, count):
    """Predictions that go straight into a shared FP32 batch are those that go there by way of rows (FP64
    batches take that route): the same sums in the same order, one affine map, so equal to 1e-6 of the largest
    (2^-23 each for the sum, the product and the shift).  One training step moves every parameter as Adam
    does from the gradient it leaves, to 1e-5 of lr and the rounding of the parameter."""
    problem_ = rt.Problem(ctx, problem_dirs[problem])
    b32 = rt.Batch(ctx, [problem_] * count, rt.F32, shared=True)
    b64 = rt.Batch(ctx, [problem_] * count, rt.F64, shared=True)
    n, nx = problem_.n_iter, problem_.nx
    mlp = rt.WarmStartMLP(ctx, nx, n, hidden=hidden, layers=layers, seed=5)
    rng = np.random.default_rng(count)
    x0 = rng.standard_normal((count, nx))
    mlp.set_normalization(np.zeros(nx), np.full(nx, 0.5), rng.standard_normal(n), 0.1 + rng.random(n))
    mlp.predict(x0, b64)
    mlp.predict(x0, b32)
    want, got = b64.iterates(), b32.iterates()
    assert np.max(np.abs(got - want)) <= 1e-6 * np.max(np.abs(want))
    # rows of the batch as the training set, one step with all of them
    mlp.dataset(b32, x0)
    before = mlp.params().astype(np.float64)
    loss = mlp.train(1, minibatch=count, lr=1e-3, seed=2)
    after, g = mlp.params().astype(np.float64), mlp.grads().astype(np.float64)
    assert np.isfinite(loss[0])
    want = before - 1e-3 * g / (np.abs(g) + 1e-8)
    assert np.max(np.abs(g)) > 0
    assert np.all(np.abs(after - want) <= 1e-8 + 2.0 ** -23 * np.abs(before))
