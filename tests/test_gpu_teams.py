"""Teams of waves in the dynamics projection: every team size a block and grid allow (1, 2, 4, 8; blocks
whose wave count is odd or not a power of two), children fewer and more than members and than a team can
take, single children (where another member takes half the node's work), dims in both row classes, affine
dynamics, and both solvers of the input systems.  Iterates after two outer iterations agree with the FP64
CPU oracle to 1e-9 (the bound of the fixed-iteration tests), and the grid barrier holds from run to run:
a second solve gives the same bits."""
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


@pytest.fixture(scope="module")
def folders(tmp_path_factory, problem_dirs):
    out = {"mid": problem_dirs["mid"], "affine": problem_dirs["affine"]}
    for events, horizon, nx, nu in ((2, 4, 5, 3), (3, 3, 65, 5), (5, 2, 9, 17), (9, 2, 3, 2), (4, 2, 70, 64), (15, 2, 2, 1)):
        d = str(tmp_path_factory.mktemp("tree"))
        configs.generate("large", d, events=events, horizon=horizon, nx=nx, nu=nu)
        out[events] = d
    return out


@pytest.mark.parametrize("workgroups,block", [(1, 64), (1, 192), (1, 384), (1, 512), (2, 128), (3, 256), (9, 512), (60, 320),
                                              (130, 256)])
@pytest.mark.parametrize("tree", ["mid", "affine", 2, 3, 4, 5, 9, 15])
def test_teams_match_oracle(ctx, folders, tree, workgroups, block):
    o = Oracle(folders[tree])
    x0 = 0.1 * configs.initial_states(3, o.nx, 1, "uniform")[0]
    ref = o.solve(x0, tol_abs=1e-30, max_iters=2, check_period=2)
    b = rt.Batch(ctx, [rt.Problem(ctx, folders[tree])], rt.F64)
    b.set_workgroups(workgroups)
    b.set_x0([x0])
    for inverse in (1, 0):
        runs = []
        for _ in range(2):
            b.reset()
            b.solve(rt.options(tol_abs=1e-30, max_iters=2, check_period=2, block_size=block, dyn_inverse=inverse))
            b.results()
            runs.append(b.iterate(0))
        assert rel_err(runs[0], ref["z"]) < 1e-9
        assert np.array_equal(runs[0], runs[1])
