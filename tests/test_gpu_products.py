"""The fused engine's per-node products at the edges of their column blocks (8), chunks (64) and row
classes (64, 128, 256): T, L, L* and the [L*; L] reductions of i.i.d. polyhedral trees (2 events, horizon 2)
against the FP64 CPU oracle, with one workgroup and with three cooperating ones.  The products sum
in the oracle's column order, so operators agree to FP64 rounding (1e-12, as in test_gpu_parity.py).
"""
import numpy as np
import pytest

from conftest import rel_err
from oracle.oracle import Oracle
from spock_amd import runtime as rt
from spock_amd.api import configs

pytestmark = pytest.mark.gpu


@pytest.fixture(scope="module")
def ctx():
    return rt.Context(0)


@pytest.mark.parametrize("workgroups", [1, 3])
@pytest.mark.parametrize("nx,nu", [(1, 1), (4, 3), (7, 8), (9, 17), (31, 1), (32, 33), (63, 2), (64, 64), (65, 5), (128, 64)])
def test_operators_at_block_edges(ctx, tmp_path, nx, nu, workgroups):
    configs.generate("large", str(tmp_path), events=2, horizon=2, nx=nx, nu=nu)
    o = Oracle(str(tmp_path))
    b = rt.Batch(ctx, [rt.Problem(ctx, str(tmp_path))], rt.F64)
    b.set_workgroups(workgroups)
    rng = np.random.default_rng(7)
    z, y = 2.0 * rng.standard_normal(o.n_iter), rng.standard_normal(o.n_iter)
    iv0 = o.n_prim + o.sI + o.sII + o.sIII
    for v in (z, y):  # entries the operators define as zero
        v[o.sU + o.sX + o.sY] = 0.0
        v[iv0:iv0 + nx + nu + 2] = 0.0
    x0 = 0.1 * rng.standard_normal(nx)
    b.set_x0([x0])
    assert rel_err(b.debug_op(rt.OP_L, z)[0][o.n_prim:], o.L(z[:o.n_prim])) < 1e-12
    assert rel_err(b.debug_op(rt.OP_LADJ, z)[0][:o.n_prim], o.Ladj(z[o.n_prim:])) < 1e-12
    assert rel_err(b.debug_op(rt.OP_T, z)[0], o.T(o.scaled_x0(x0), z)) < 1e-12
    _, sc = b.debug_op(rt.OP_ELL, z, y)
    ref = o.dotM(z, y)
    ell = np.concatenate([o.Ladj(y[o.n_prim:]), o.L(y[:o.n_prim])])
    assert abs(sc[0] - ref) <= 1e-12 * max(1.0, float(np.abs(z) @ np.abs(y)))
    assert abs(sc[1] - np.max(np.abs(y / o.gamma - ell))) <= 1e-12 * np.max(np.abs(y / o.gamma))
