"""One batch solved with changing numbers of workgroups, from fewer than the grid barrier has groups to more and
back: every solve gives the bits that a new batch gives with that number, and the autotuner runs on a
batch last solved by a few."""
import numpy as np
import pytest

from spock_amd import runtime as rt
from spock_amd.api import configs

pytestmark = pytest.mark.gpu

OPTS = dict(tol_abs=1e-30, max_iters=4, check_period=2)


@pytest.fixture(scope="module")
def ctx():
    return rt.Context(0)


def solved(batch, x0, workgroups, **kw):
    batch.set_workgroups(workgroups)
    batch.set_x0([x0])
    batch.reset()
    batch.solve(rt.options(**OPTS, **kw))
    batch.results()
    return batch.iterate(0)


@pytest.mark.parametrize("dtype", [rt.F64, rt.F32])
@pytest.mark.parametrize("counts", [(4, 32), (32, 4, 32), (2, 3, 8, 256, 7, 9), (3, 9, 1, 5, 64, 2, 130)],
                         ids=lambda c: "-".join(map(str, c)))
def test_counts_change(ctx, problem_dirs, counts, dtype):
    p = rt.Problem(ctx, problem_dirs["mid"])
    x0 = 0.1 * configs.initial_states(3, p.nx, 1, "uniform")[0]
    b = rt.Batch(ctx, [p], dtype)
    for n in counts:
        print("workgroups", n, flush=True)
        z = solved(b, x0, n)
        assert np.all(np.isfinite(z))
        assert np.array_equal(z, solved(rt.Batch(ctx, [p], dtype), x0, n)), n


def test_autotune_after_a_few(ctx, problem_dirs):
    p = rt.Problem(ctx, problem_dirs["mid"])
    x0 = 0.1 * configs.initial_states(3, p.nx, 1, "uniform")[0]
    b = rt.Batch(ctx, [p], rt.F64)
    solved(b, x0, 5)
    best, table = b.autotune_workgroups(rt.options(**OPTS), iters=4)
    assert best in table
    assert np.array_equal(solved(b, x0, 6), solved(rt.Batch(ctx, [p], rt.F64), x0, 6))
