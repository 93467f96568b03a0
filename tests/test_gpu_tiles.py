"""The tile engine's node operators at the edges of their row tiles (16, 32 and 64 rows at a time) and column
groups (16): T, L, L*, the projections and the [L*; L] reductions of 17 instances (one full workgroup and one with
a single instance) on polyhedral trees of 2 events and horizon 2, against the FP64 CPU oracle.  FP64 sums follow
the oracle's up to their order: 1e-12, as in test_gpu_shared.py.  FP32: each sum of up to K terms errs
by K 2^-24 of its magnitudes at most, with K <= nx + nu + 2 and a chain of four products in the dynamics, whose
magnitudes stay within 16 times the largest entry: 4 * 16 * (nx + nu + 2) * 2^-24 of it."""
import numpy as np
import pytest

from conftest import rel_err
from oracle.oracle import Oracle
from spock_amd import runtime as rt
from spock_amd.api import configs

pytestmark = pytest.mark.gpu

COUNT = 17


@pytest.fixture(scope="module")
def ctx():
    return rt.Context(0)


@pytest.mark.parametrize("nx,nu", [(1, 1), (15, 16), (16, 15), (17, 17), (31, 32), (32, 31), (33, 1), (63, 2), (64, 32),
                                   (65, 16), (128, 5)])
@pytest.mark.parametrize("engine,dtype", [(17, rt.F64), (16, rt.F64), (17, rt.F32)])
def test_operators_at_tile_edges(ctx, tmp_path, nx, nu, engine, dtype):
    configs.generate("large", str(tmp_path), events=2, horizon=2, nx=nx, nu=nu)
    o = Oracle(str(tmp_path))
    p = rt.Problem(ctx, str(tmp_path))
    b = rt.Batch(ctx, [p] * COUNT, dtype, shared=True, engine=engine)
    tol = 1e-12 if dtype == rt.F64 else 4 * 16 * (nx + nu + 2) * 2.0 ** -24
    rng = np.random.default_rng(nx + nu)
    z, y = rng.standard_normal((COUNT, o.n_iter)), rng.standard_normal((COUNT, o.n_iter))
    iv0 = o.n_prim + o.sI + o.sII + o.sIII
    for v in (z, y):  # entries the operators define as zero
        v[:, o.sU + o.sX + o.sY] = 0.0
        v[:, iv0:iv0 + nx + nu + 2] = 0.0
    if dtype == rt.F32:
        z, y = z.astype(np.float32).astype(np.float64), y.astype(np.float32).astype(np.float64)
    x0 = 0.1 * rng.standard_normal((COUNT, nx))
    b.set_x0(list(x0))
    Z = z.ravel()
    L = b.debug_op(rt.OP_L, Z)[0].reshape(COUNT, -1)
    La = b.debug_op(rt.OP_LADJ, Z)[0].reshape(COUNT, -1)
    T = b.debug_op(rt.OP_T, Z)[0].reshape(COUNT, -1)
    sc = b.debug_op(rt.OP_ELL, Z, y.ravel())[1]
    for k in range(COUNT):
        assert rel_err(L[k][o.n_prim:], o.L(z[k][:o.n_prim])) < tol
        assert rel_err(La[k][:o.n_prim], o.Ladj(z[k][o.n_prim:])) < tol
        assert rel_err(T[k], o.T(o.scaled_x0(x0[k]), z[k])) < tol
        ell = np.concatenate([o.Ladj(y[k][o.n_prim:]), o.L(y[k][:o.n_prim])])
        assert abs(sc[2 * k] - o.dotM(z[k], y[k])) <= tol * max(1.0, float(np.abs(z[k]) @ np.abs(y[k])))
        assert abs(sc[2 * k + 1] - np.max(np.abs(y[k] / o.gamma - ell))) <= tol * np.max(np.abs(y[k] / o.gamma))
