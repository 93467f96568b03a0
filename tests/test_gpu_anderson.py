"""The tree-reduced Householder least squares of the fused engine for every Anderson memory it is built
for (1 to 8), with one workgroup and spread over several (70 leaves lanes of the workgroup stage with two
triangles each), against the FP64 CPU oracle's column-by-column Householder QR.

Iterates after m + 4 outer iterations, the first few with a least squares in them, agree to 1e-9 (the
bound of the fixed-iteration tests) with identical SuperMann branch counts."""
import pytest

from conftest import rel_err
from oracle.oracle import Oracle
from spock_amd import runtime as rt
from spock_amd.api import configs

pytestmark = pytest.mark.gpu


@pytest.fixture(scope="module")
def ctx():
    return rt.Context(0)


@pytest.mark.parametrize("workgroups", [1, 3, 70])
@pytest.mark.parametrize("m", [1, 2, 3, 4, 5, 6, 7, 8])
def test_anderson_memories_match_oracle(ctx, problem_dirs, m, workgroups):
    d = problem_dirs["small"]
    o = Oracle(d)
    x0 = configs.initial_states(1, o.nx, 1, "uniform")[0]
    iters = m + 4
    ref = o.solve(x0, tol_abs=1e-30, max_iters=iters, check_period=iters, anderson=m)
    b = rt.Batch(ctx, [rt.Problem(ctx, d)], rt.F64)
    b.set_workgroups(workgroups)
    b.set_x0([x0])
    b.solve(rt.options(tol_abs=1e-30, max_iters=iters, check_period=iters, anderson_buffer=m))
    r = b.results()[0][0]
    assert (r["iters"], r["k0"], r["k1"], r["k2"], r["k2bt"], r["k3"]) == \
        (ref["iters"], ref["k0"], ref["k1"], ref["k2"], ref["k2bt"], ref["k3"])
    assert rel_err(b.iterate(0), ref["z"]) < 1e-9
