"""Performance cases of the solver: what a user's program has it do, through the Python binding.

Four kinds of work, each a sequence of the calls that a program makes between two of its own steps:

  single   one problem, one solve: the drop-in ``Cache`` use (receding-horizon control of one plant).
           A pass sets the initial state, clears the iterate, solves and reads status and solution.
  uneven   one batch of many different trees, solved by one persistent launch.
  shared   many initial states of one problem in lockstep: cold solves, FP32 bulk solves warm-started
           from device rows (a predicted or previous solution), FP64 polish of FP32 solutions.
  predict / train   the learned warm start: predictions written into a batch, and Adam training.

Solves run a fixed number of outer iterations (tolerance 0), so every pass does the same work.  FP32
SPOCK solves run few of them (5; 10 on the 229-node plant; 3 with polyhedral constraints): SuperMann
with Anderson directions amplifies rounding from iteration to iteration, and beyond that two orders
of summation are no longer comparable.  The plain CP method does not amplify it.

Problems come from the package's seeded generators and are made once per process, as a program loads
its plant model once; initial states, starting iterates, network weights and training targets come
from the seed.  ``exact`` restates the iteration and the network in plain torch in 64 bits, from the
generated problem files.
"""
import functools
import importlib.util
import json
import math
import os
import sys
import tempfile

import numpy as np
import torch

ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))


def _package():
    """The package (its folder's name holds a dot) as ``spock_amd``, from the tree that this file is in."""
    if "spock_amd" not in sys.modules:
        folder = os.path.join(ROOT, "spock.cu_amd")
        spec = importlib.util.spec_from_file_location("spock_amd", os.path.join(folder, "__init__.py"),
                                                      submodule_search_locations=[folder])
        module = importlib.util.module_from_spec(spec)
        sys.modules["spock_amd"] = module
        spec.loader.exec_module(module)
    from spock_amd import runtime
    from spock_amd.api import configs
    return runtime, configs


# ------------------------------------------------------------------------------------- the cases
def listed():
    return [
        # The smallest call: the 31-node plant (nx=3, nu=2) in FP64, one control step's iterations.
        dict(name="single_31node_f64", kind="single", problem="small", dtype="f64", method="spock", iters=50,
             workgroups=1, ls="householder"),
        # The drop-in's usual problem at the size of its reference drivers: 229 nodes, nx=50, nu=20, as the C ABI
        # runs it by default (one workgroup) and as the drop-in runs it (32 workgroups).
        dict(name="single_229node_f64", kind="single", problem="mid", dtype="f64", method="spock", iters=25,
             workgroups=1, ls="householder"),
        dict(name="single_229node_f64_32wg", kind="single", problem="mid", dtype="f64", method="spock", iters=50,
             workgroups=32, ls="householder"),
        # The reference's server air-conditioning plant (63 nodes, nx=nu=50) with the plain CP method, FP32.
        dict(name="single_server_f32_cp", kind="single", problem="server5", dtype="f32", method="cp", iters=50,
             workgroups=1, ls="householder"),
        # Large trees with polyhedral constraints and linear costs (nx=100, nu=40), spread over the GPU: 341 nodes in
        # FP64, 1365 nodes in FP32.
        dict(name="single_341node_f64_128wg", kind="single", problem="poly100x40h4", dtype="f64", method="spock",
             iters=15, workgroups=128, ls="householder"),
        dict(name="single_1365node_f32_256wg_cp", kind="single", problem="poly100x40h5", dtype="f32", method="cp",
             iters=10, workgroups=256, ls="householder"),
        # Different plants in one launch: 256 instances of 64 uneven trees, FP32 bulk with the Gram least squares.
        dict(name="uneven_256_f32", kind="uneven", trees=64, first=0, count=256, dtype="f32", method="spock",
             iters=5, ls="gram"),
        # Serving: 4,096 initial states of the 229-node plant, FP32 bulk, warm-started from predicted rows.
        dict(name="shared_4096_f32_warm", kind="shared", problem="mid", dtype="f32", method="spock", iters=10,
             count=4096, warm=True),
        # The FP64 polish of a batch of FP32 solutions.
        dict(name="shared_1000_f64_warm", kind="shared", problem="mid", dtype="f64", method="spock", iters=5,
             count=1000, warm=True),
        # A small fleet on the small plant, cold, an odd count, plain CP in FP64.
        dict(name="shared_70_small_f64_cp", kind="shared", problem="small", dtype="f64", method="cp", iters=50,
             count=70, warm=False),
        # The learned warm start for a whole serving batch, and a short training run on one batch of solutions.
        dict(name="predict_4096", kind="predict", problem="mid", count=4096, hidden=512, layers=3),
        dict(name="train_256", kind="train", problem="mid", count=256, hidden=512, layers=3, epochs=40),
    ]


def _log_int(rng, lo, hi):
    return int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))


def _bounded(problem, dtype, method, iters):
    """FP32 SPOCK with polyhedral constraints is compared over 3 iterations only (see above)."""
    return min(iters, 3) if problem.startswith("poly") and dtype == "f32" and method == "spock" else iters


def draw(rng):
    kind = rng.choice(["single", "single", "single", "uneven", "shared", "shared", "shared", "predict", "train"])
    dtype = rng.choice(["f64", "f32"])
    method = rng.choice(["spock", "spock", "cp"])
    iters = rng.randint(5, 50) if dtype == "f64" else rng.randint(5, 10) if method == "cp" else rng.randint(3, 5)
    if kind == "single":
        problem = rng.choice(["small", "mid", "affine", "nocon", "server%d" % rng.randint(2, 5),
                              "uneven%d" % rng.randint(100, 400),
                              "poly%dx%dh%d" % (rng.randint(4, 100), rng.randint(2, 40), rng.randint(2, 4))])
        workgroups = 1 if problem in ("small", "affine", "nocon") else rng.choice([1, 1, _log_int(rng, 2, 256)])
        return dict(kind=kind, problem=problem, dtype=dtype, method=method,
                    iters=_bounded(problem, dtype, method, iters), workgroups=workgroups,
                    ls=rng.choice(["householder", "gram"]))
    if kind == "uneven":
        trees = rng.randint(2, 32)
        return dict(kind=kind, trees=trees, first=rng.randint(64, 400), count=trees * rng.randint(1, 10), dtype=dtype,
                    method=method, iters=min(iters, 20), ls=rng.choice(["householder", "gram"]))
    if kind == "shared":
        problem = rng.choice(["small", "mid", "mid", "nocon", "affine", "uneven%d" % rng.randint(100, 400),
                              "poly%dx%dh%d" % (rng.randint(4, 40), rng.randint(2, 20), rng.randint(2, 3))])
        return dict(kind=kind, problem=problem, dtype=dtype, method=method,
                    iters=_bounded(problem, dtype, method, min(iters, 10)),
                    count=_log_int(rng, 3, 4096 if dtype == "f32" else 1024), warm=rng.random() < 0.5)
    problem = rng.choice(["small", "mid", "uneven%d" % rng.randint(100, 400)])
    hidden, layers = rng.choice([64, 128, 256, 512, 200]), rng.randint(1, 3)
    if kind == "predict":
        return dict(kind=kind, problem=problem, count=_log_int(rng, 16, 4096), hidden=hidden, layers=layers)
    return dict(kind=kind, problem=problem, count=_log_int(rng, 30, 256), hidden=hidden, layers=layers,
                epochs=rng.randint(5, 40))


# ------------------------------------------------------------------------------------- problems
_FOLDERS = {}


def _folder(problem):
    """The generated problem files of a plant, made once per process."""
    if problem not in _FOLDERS:
        _, configs = _package()
        holder = tempfile.TemporaryDirectory(prefix="spock_perf_")
        if problem.startswith("server"):
            configs.generate("server", holder.name, horizon=int(problem[6:]))
        elif problem.startswith("uneven"):
            configs.uneven_instance(holder.name, int(problem[6:]))
        elif problem.startswith("poly"):
            nx, rest = problem[4:].split("x")
            nu, horizon = rest.split("h")
            configs.generate("large", holder.name, nx=int(nx), nu=int(nu), horizon=int(horizon))
        else:
            configs.generate(problem, holder.name)
        _FOLDERS[problem] = holder
    return _FOLDERS[problem].name


@functools.lru_cache(maxsize=None)
def _context():
    runtime, _ = _package()
    return runtime.Context(0)


@functools.lru_cache(maxsize=None)
def _loaded(problem):
    runtime, _ = _package()
    return runtime.Problem(_context(), _folder(problem))


@functools.lru_cache(maxsize=None)
def _sizes(problem):
    with open(os.path.join(_folder(problem), "data.json")) as fh:
        info = json.load(fh)
    return info["numStates"], info["numInputs"]


def _initial_states(problem, seed, count):
    """Initial states of the plant's operating range (the scale that its constraints can serve)."""
    nx, _ = _sizes(problem)
    rng = np.random.default_rng([seed, 17])
    if problem.startswith("poly"):
        return 0.05 * rng.standard_normal((count, nx))
    if problem.startswith("server"):
        return 0.1 + 0.05 * rng.standard_normal((count, nx))
    if problem in ("small", "affine", "nocon"):
        return rng.uniform(-1.0, 1.0, (count, nx))
    return 0.5 * rng.standard_normal((count, nx))


def _instances(case):
    """Problem name of every instance of a solve case, in order."""
    if case["kind"] == "uneven":
        return ["uneven%d" % (case["first"] + k % case["trees"]) for k in range(case["count"])]
    return [case["problem"]] * case.get("count", 1)


def _case_states(case, seed):
    names = _instances(case)
    if case["kind"] != "uneven":
        return _initial_states(case["problem"], seed, len(names))
    return [_initial_states(name, seed * 1000 + k, 1)[0] for k, name in enumerate(names)]


def _rows(case, seed, n):
    """Starting iterates as a predictor leaves them in device memory: FP32 rows."""
    gen = torch.Generator(device="cuda").manual_seed(seed)
    return 0.1 * torch.randn((case["count"], n), generator=gen, device="cuda", dtype=torch.float32)


def _network(case, seed):
    """Flat FP32 parameters (per layer W row-major, then b) and the output normalization."""
    n_in, n_out = _sizes(case["problem"])[0], _loaded(case["problem"]).n_iter
    dims = [n_in] + [case["hidden"]] * case["layers"] + [n_out]
    rng = np.random.default_rng([seed, 23])
    parts = []
    for a, b in zip(dims[:-1], dims[1:]):
        parts.append((rng.uniform(-1.0, 1.0, a * b) * math.sqrt(3.0 / a)).astype(np.float32))
        parts.append((0.05 * rng.standard_normal(b)).astype(np.float32))
    scale = (0.05 + rng.random(n_out)).astype(np.float32)
    shift = rng.standard_normal(n_out).astype(np.float32)
    return dims, np.concatenate(parts), scale, shift


# ------------------------------------------------------------------------------------- prepare / run
def prepare(case, seed):
    runtime, _ = _package()
    ctx = _context()
    dtype = runtime.F32 if case.get("dtype") == "f32" else runtime.F64
    if case["kind"] in ("single", "uneven", "shared"):
        problems = [_loaded(name) for name in _instances(case)]
        state = dict(kind=case["kind"], x0=_case_states(case, seed), f32=case["dtype"] == "f32",
                     batch=runtime.Batch(ctx, problems, dtype, shared=case["kind"] == "shared"))
        state["opts"] = runtime.options(
            tol_abs=0.0, max_iters=case["iters"], check_period=case["iters"],
            method=runtime.CP if case["method"] == "cp" else runtime.SPOCK,
            ls_method=runtime.LS_GRAM if case.get("ls") == "gram" else runtime.LS_HOUSEHOLDER)
        if case["kind"] == "single":
            state["batch"].set_workgroups(case["workgroups"])
        if case["kind"] == "shared":
            n = problems[0].n_iter
            state["rows"] = _rows(case, seed, n) if case["warm"] else None
            state["out"] = torch.empty((case["count"], n), device="cuda", dtype=torch.float32)
        return state
    dims, params, scale, shift = _network(case, seed)
    mlp = runtime.WarmStartMLP(ctx, dims[0], dims[-1], hidden=case["hidden"], layers=case["layers"], seed=seed)
    mlp.set_params(params)
    x0 = _initial_states(case["problem"], seed, case["count"])
    batch = runtime.Batch(ctx, [_loaded(case["problem"])] * case["count"], runtime.F32, shared=True)
    state = dict(kind=case["kind"], mlp=mlp, batch=batch, x0=x0)
    if case["kind"] == "predict":
        mlp.set_normalization(np.zeros(dims[0], np.float32), np.full(dims[0], 0.5, np.float32), shift, scale)
        state["out"] = torch.empty((case["count"], dims[-1]), device="cuda", dtype=torch.float32)
        return state
    # the training set: solved iterates of the batch's initial states, here rows of their kind
    rows = _targets(case, seed, dims[-1])
    torch.cuda.synchronize()
    batch.set_iterates_device(rows.data_ptr(), dims[-1])
    mlp.dataset(batch, x0)
    state.update(epochs=case["epochs"], minibatch=case["count"])
    return state


def _targets(case, seed, n):
    """Solutions vary smoothly with the initial state: a nonlinear map of it plus a little noise."""
    gen = torch.Generator(device="cuda").manual_seed(seed)
    x0 = torch.tensor(_initial_states(case["problem"], seed, case["count"]), dtype=torch.float32, device="cuda")
    w = torch.randn((x0.shape[1], n), generator=gen, device="cuda") / math.sqrt(x0.shape[1])
    noise = torch.randn((case["count"], n), generator=gen, device="cuda")
    return torch.tanh((x0[:, :, None] * w[None]).sum(1) if x0.numel() * n < 1 << 28 else x0 @ w) + 0.05 * noise


def run(state):
    batch = state["batch"]
    if state["kind"] == "predict":
        state["mlp"].predict(state["x0"], batch)
        batch.get_iterates_device(state["out"].data_ptr(), state["out"].shape[1])
        return state["out"]
    if state["kind"] == "train":
        losses = state["mlp"].train(state["epochs"], minibatch=state["minibatch"], lr=1e-4, seed=1)
        return {"loss": losses, "params": state["mlp"].params()}
    rows = state.get("rows")
    batch.set_x0(state["x0"])
    if rows is not None:
        batch.set_iterates_device(rows.data_ptr(), rows.shape[1])
    else:
        batch.reset()
    batch.solve(state["opts"], warm=rows is not None)
    results, _ = batch.results()
    if state["kind"] == "shared":
        batch.get_iterates_device(state["out"].data_ptr(), state["out"].shape[1])
        z = state["out"]
    else:
        z = batch.iterates()
        z = z.astype(np.float32) if state["f32"] else z
    return {"z": z, "iters": np.array([r["iters"] for r in results]), "status": np.array([r["status"] for r in results])}


# ------------------------------------------------------------------------------------- work
def work(case):
    """Bytes and operations of one pass.  Solves: per outer iteration T reads the iterate and writes its
    image, and SuperMann also reads the previous iterate and residual and two older columns of each Anderson
    history and writes the residual, the new columns and the next iterate; the distinct matrices are read
    once per iteration, and the products are those of T (L*, the dynamics sweeps, the kernel projections, L)
    and of one more L* for SuperMann's norm.  The network: parameters, inputs and outputs (training: the
    parameters, gradients and moments of each step)."""
    if case["kind"] in ("predict", "train"):
        nx, _ = _sizes(case["problem"])
        n = _Plant(case["problem"], "cpu").n
        dims = [nx] + [case["hidden"]] * case["layers"] + [n]
        weights = sum(a * b for a, b in zip(dims[:-1], dims[1:]))
        if case["kind"] == "predict":
            return {"bytes": 2 * weights + case["count"] * (8 * nx + 4 * n), "flops": 2 * weights * case["count"]}
        return {"bytes": case["epochs"] * (28 * weights + 8 * case["count"] * n),
                "flops": case["epochs"] * 6 * weights * case["count"]}
    word = 4 if case["dtype"] == "f32" else 8
    spock = case["method"] == "spock"
    names = _instances(case)
    bytes_, flops = 0.0, 0.0
    for name in sorted(set(names)):
        plant, count = _Plant(name, "cpu"), names.count(name)
        steps = case["iters"] + 1
        bytes_ += steps * word * ((12 if spock else 2) * plant.n * count + plant.distinct)
        flops += steps * 2.0 * count * (plant.products + (plant.adjoint if spock else 0))
    return {"bytes": bytes_, "flops": flops}


# ------------------------------------------------------------------------------------- exact
def _read(folder, name):
    """A tensor file as (matrices, rows, columns) in 64 bits; None if the problem has none."""
    path = os.path.join(folder, name + ".bt")
    if not os.path.isfile(path):
        return None
    with open(path, "rb") as fh:
        r, c, m = (int(v) for v in np.fromfile(fh, dtype="<u8", count=3))
        data = np.fromfile(fh, dtype="<u8" if name.endswith("_u") else "<f8", count=r * c * m)
    return data.reshape(m, c, r).transpose(0, 2, 1)


class _Plant:
    """One problem's data in 64 bits and the operators of the iteration on rows of instances."""

    def __init__(self, problem, device):
        folder = _folder(problem)
        with open(os.path.join(folder, "data.json")) as fh:
            info = json.load(fh)
        self.N, self.nl, self.E = info["numNodes"], info["numNonleafNodes"], info["numEvents"]
        self.nx, self.nu, self.yD = info["numStates"], info["numInputs"], 2 * info["numEvents"] + 1
        self.nlf, self.gamma, self.stages = self.N - self.nl, info["stepSize"], info["numStages"]
        self.affine = info["dynamics"]["type"] == "affine"
        N, nl, nx, nu = self.N, self.nl, self.nx, self.nu

        def table(name):
            v = _read(folder, name + "_d")
            return None if v is None else torch.tensor(np.ascontiguousarray(v), device=device)

        def ints(name):
            return torch.tensor(_read(folder, name + "_u").reshape(-1).astype(np.int64), device=device)

        self.anc, self.first, self.kids = ints("ancestors"), ints("childrenFrom"), ints("numChildren")
        self.stage_from, self.stage_to = ints("stageFrom").tolist(), ints("stageTo").tolist()
        self.anc[0] = 0
        self.con3 = self.con5 = 0
        self.con = []
        for part, nodes in (("nonleafConstraint", nl), ("leafConstraint", self.nlf)):
            G = table(part + "Gamma")
            lo, hi = (table(part + "ILB"), table(part + "IUB")) if G is None else (table(part + "GLB"), table(part + "GUB"))
            if lo is not None:
                lo, hi = (v.reshape(1, -1).repeat(nodes, 1) for v in (lo, hi))
                if G is None and nodes == nl:  # a box leaves the root's state free
                    lo[0, :nx], hi[0, :nx] = -math.inf, math.inf
            self.con.append((None if G is None else G[0], lo, hi))
        self.con3 = 0 if self.con[0][1] is None else self.con[0][1].shape[1]
        self.con5 = 0 if self.con[1][1] is None else self.con[1][1].shape[1]
        prim = [nu * nl, nx * N, self.yD * nl, N, N]
        dual = [self.yD * nl, nl, self.con3 * nl, (nx + nu + 2) * N, self.con5 * self.nlf, (nx + 2) * self.nlf]
        self.split_prim, self.split_dual = prim, dual
        self.n_prim, self.n = sum(prim), sum(prim) + sum(dual)
        rows3, rows5 = (self.con3 if self.con[0][0] is not None else 0), (self.con5 if self.con[1][0] is not None else 0)
        self.adjoint = (N - 1) * (nx * nx + nu * nu) + self.nlf * nx * nx + nl * rows3 * (nx + nu) + self.nlf * rows5 * nx
        sweeps = (N - 1) * (2 * nx * nx + 3 * nx * nu) + nl * (2 * nx * nu + nu * nu) + nl * (4 * self.E + 1) ** 2
        self.products = 2 * self.adjoint + sweeps
        self.distinct = self.E * (2 * nx * nx + 3 * nx * nu) * self.stages + nx * nx + rows3 * (nx + nu) + rows5 * nx
        if device == "cpu":
            return  # sizes only
        self.BTr, self.AB, self.K = table("dynamics_BTr"), table("dynamics_AB"), table("dynamics_K")
        self.ABKTr, self.APB = table("dynamics_ABKTr"), table("dynamics_APB")
        low = table("dynamics_lowCholesky")
        self.RtInv = torch.linalg.inv(low @ low.transpose(1, 2))
        if self.affine:
            self.e = table("dynamics_c").reshape(N, nx)
            self.Pe = (table("dynamics_P") @ self.e[:, :, None])[:, :, 0]
        self.NN, self.b = table("risk_NNtr"), table("risk_b").reshape(nl, self.yD)
        self.sQ, self.sR = table("nonleafCost_sqrtQ"), table("nonleafCost_sqrtR")
        self.trans = table("nonleafCost_translation").reshape(N, -1)
        self.lsQ, self.ltrans = table("leafCost_sqrtQ")[0], table("leafCost_translation").reshape(-1)
        q, r, lq = table("nonleafCost_q"), table("nonleafCost_r"), table("leafCost_q")
        self.q = torch.zeros((N, nx), dtype=torch.float64, device=device) if q is None else q.reshape(N, nx)
        self.r = torch.zeros((N, nu), dtype=torch.float64, device=device) if r is None else r.reshape(N, nu)
        self.lq = torch.zeros(nx, dtype=torch.float64, device=device) if lq is None else lq.reshape(-1)
        scaling = table("scaling")
        self.scaling = None if scaling is None else scaling.reshape(-1)[:nx]

    def prim(self, p):
        u, x, y, t, s = torch.split(p, self.split_prim, dim=1)
        B = p.shape[0]
        return u.reshape(B, self.nl, self.nu), x.reshape(B, self.N, self.nx), y.reshape(B, self.nl, self.yD), t, s

    def dual(self, d):
        I, II, III, IV, V, VI = torch.split(d, self.split_dual, dim=1)
        B = d.shape[0]
        return (I.reshape(B, self.nl, self.yD), II, III.reshape(B, self.nl, self.con3), IV.reshape(B, self.N, -1),
                V.reshape(B, self.nlf, self.con5), VI.reshape(B, self.nlf, -1))

    @staticmethod
    def mul(M, v):
        """Per-node products: M (nodes, r, c), v (B, nodes, c)."""
        return (M @ v.permute(1, 2, 0)).permute(2, 0, 1)

    def L(self, p):
        u, x, y, t, s = self.prim(p)
        B, nl = p.shape[0], self.nl
        xu = torch.cat([x[:, :nl], u], 2)
        out = [y, s[:, :nl] - (y * self.b).sum(2)]
        G, lo, _ = self.con[0]
        out.append(xu if G is None else xu @ G.T) if lo is not None else None
        xa, ua = x[:, self.anc], u[:, self.anc]
        h = 0.5 * (t - (xa * self.q).sum(2) - (ua * self.r).sum(2))
        IV = torch.cat([self.mul(self.sQ, xa), self.mul(self.sR, ua), h[:, :, None], h[:, :, None]], 2)
        IV[:, 0] = 0
        out.append(IV)
        xl = x[:, nl:]
        G, lo, _ = self.con[1]
        out.append(xl if G is None else xl @ G.T) if lo is not None else None
        h = 0.5 * (s[:, nl:] - xl @ self.lq)
        out.append(torch.cat([xl @ self.lsQ.T, h[:, :, None], h[:, :, None]], 2))
        return torch.cat([v.reshape(B, -1) for v in out], 1)

    def adj(self, d):
        I, II, III, IV, V, VI = self.dual(d)
        B, nl, nx, nu = d.shape[0], self.nl, self.nx, self.nu
        u, x = d.new_zeros(B, nl, nu), d.new_zeros(B, self.N, nx)
        G, lo, _ = self.con[0]
        if lo is not None:
            xu = III if G is None else III @ G
            x[:, :nl] += xu[:, :, :nx]
            u += xu[:, :, nx:]
        ab = IV[:, :, -2] + IV[:, :, -1]
        cx = self.mul(self.sQ.transpose(1, 2), IV[:, :, :nx]) - 0.5 * ab[:, :, None] * self.q
        cu = self.mul(self.sR.transpose(1, 2), IV[:, :, nx:nx + nu]) - 0.5 * ab[:, :, None] * self.r
        x.index_add_(1, self.anc[1:], cx[:, 1:])
        u.index_add_(1, self.anc[1:], cu[:, 1:])
        G, lo, _ = self.con[1]
        if lo is not None:
            x[:, nl:] += V if G is None else V @ G
        lab = VI[:, :, -2] + VI[:, :, -1]
        x[:, nl:] += VI[:, :, :nx] @ self.lsQ - 0.5 * lab[:, :, None] * self.lq
        t = 0.5 * ab
        t[:, 0] = 0
        s = torch.cat([II, 0.5 * lab], 1)
        return torch.cat([u.reshape(B, -1), x.reshape(B, -1), (I - II[:, :, None] * self.b).reshape(B, -1), t, s], 1)

    def dynamics(self, x, u, x0):
        """Projection of (x, u) onto the dynamics from x0: the backward and the forward sweep."""
        nl = self.nl
        q, d = -x, torch.zeros_like(u)
        for stage in range(self.stages - 2, -1, -1):
            i = slice(self.stage_from[stage], self.stage_to[stage] + 1)
            j = slice(self.stage_from[stage + 1], self.stage_to[stage + 1] + 1)
            to = self.anc[j] - i.start
            qj = q[:, j] + self.Pe[j] if self.affine else q[:, j]
            e = u[:, i].index_add(1, to, -self.mul(self.BTr[j], qj))
            d[:, i] = self.mul(self.RtInv[i], e)
            if stage:
                di = d[:, i]
                sums = self.mul(self.K[i].transpose(1, 2), di - u[:, i]) - x[:, i]
                q[:, i] = sums.index_add(1, to, self.mul(self.APB[j], di[:, to]) + self.mul(self.ABKTr[j], qj))
        x, u = x.clone(), u.clone()
        x[:, 0] = x0
        for stage in range(self.stages - 1):
            i = slice(self.stage_from[stage], self.stage_to[stage] + 1)
            j = slice(self.stage_from[stage + 1], self.stage_to[stage + 1] + 1)
            u[:, i] = self.mul(self.K[i], x[:, i]) + d[:, i]
            a = self.anc[j]
            x[:, j] = self.mul(self.AB[j], torch.cat([x[:, a], u[:, a]], 2)) + (self.e[j] if self.affine else 0)
        return x, u

    def kernel(self, y, t, s):
        """Projection of each nonleaf node's (y, children's t, children's s) onto its kernel."""
        B, nl, E, yD = y.shape[0], self.nl, self.E, self.yD
        slot = torch.arange(E, device=y.device)
        has = slot[None] < self.kids[:nl, None]
        child = torch.where(has, self.first[:nl, None] + slot[None], 0)
        v = self.mul(self.NN, torch.cat([y, t[:, child] * has, s[:, child] * has], 2))
        t, s = t.clone(), s.clone()
        t[:, child[has]] = v[:, :, yD:yD + E][:, has]
        s[:, child[has]] = v[:, :, yD + E:][:, has]
        return v[:, :, :yD], t, s

    @staticmethod
    def cone(w):
        """Second-order cone projection of the rows (v, t)."""
        nrm, tl = w[..., :-1].norm(dim=-1, keepdim=True), w[..., -1:]
        half = 0.5 * (nrm + tl)
        p = torch.cat([w[..., :-1] * (half / nrm.clamp_min(1e-300)), half], -1)
        return torch.where(nrm <= tl, w, torch.where(nrm <= -tl, torch.zeros_like(w), p))

    def T(self, z, x0):
        g, B, nl = self.gamma, z.shape[0], self.nl
        zp, zd = z[:, :self.n_prim], z[:, self.n_prim:]
        u, x, y, t, s = self.prim(zp - g * self.adj(zd))
        s = s.clone()
        s[:, 0] -= g
        x, u = self.dynamics(x, u, x0)
        y, t, s = self.kernel(y, t, s)
        cp = torch.cat([u.reshape(B, -1), x.reshape(B, -1), y.reshape(B, -1), t, s], 1)
        w = (self.L(2 * cp - zp) * g + zd) / g
        I, II, III, IV, V, VI = self.dual(w)
        IV, VI = IV + self.trans, VI + self.ltrans
        free = torch.arange(self.yD, device=z.device)[None] >= 2 * self.kids[:nl, None]
        proj = [torch.where(free, I, I.clamp_min(0)), II.clamp_min(0)]
        proj.append(torch.maximum(torch.minimum(III, self.con[0][2]), self.con[0][1])) if self.con3 else None
        proj.append(self.cone(IV))
        proj.append(torch.maximum(torch.minimum(V, self.con[1][2]), self.con[1][1])) if self.con5 else None
        proj.append(self.cone(VI))
        moved = [I, II] + ([III] if self.con3 else []) + [IV] + ([V] if self.con5 else []) + [VI]
        cd = torch.cat([(a - p).reshape(B, -1) for a, p in zip(moved, proj)], 1) * g
        return torch.cat([cp, cd], 1)

    def dot(self, a, b):
        """<a, M b> of each row, M = I - gamma [0 L*; L 0]."""
        ell = torch.cat([self.adj(b[:, self.n_prim:]), self.L(b[:, :self.n_prim])], 1)
        return (a * (b - self.gamma * ell)).sum(1)

    def solve(self, x0, z, warm, method, iters, memory=3, inner=8):
        """`iters` outer iterations from rows z (FP64), then the last application of T."""
        if self.scaling is not None:
            x0 = x0 * self.scaling
        if method == "cp":
            for _ in range(iters + 1):
                z = self.T(z, x0)
            return z
        B = z.shape[0]
        zprev, rprev = (z, torch.zeros_like(z)) if warm else (torch.ones_like(z), torch.ones_like(z))
        zeta = torch.full((B,), math.inf, dtype=torch.float64, device=z.device)
        safe = zeta.clone()
        Y, S = [], []
        for it in range(iters):
            tz = self.T(z, x0)
            r = z - tz
            w = self.dot(r, r).sqrt()
            Y, S = [r - rprev] + Y[:memory - 1], [(z - zprev) - (r - rprev)] + S[:memory - 1]
            zprev, rprev = z, r
            d = -r - (self.lsq(Y, S, r) if it >= memory else 0)
            blind = w <= 0.99 * zeta
            zeta = torch.where(blind, w, zeta)
            nxt, left, tau = zprev + d, ~blind, torch.ones_like(w)
            for _ in range(inner):
                if not bool(left.any()):
                    break
                step = d * tau[:, None]
                trial = zprev + step
                rt = trial - self.T(trial, x0)
                wt = self.dot(rt, rt).sqrt()
                k1 = left & (w <= safe) & (wt <= 0.99 * w)
                rho = wt * wt - self.dot(rt, step)
                k2 = left & ~k1 & (rho >= 0.1 * wt * w)
                safe = torch.where(k1, wt + 0.99 ** it, safe)
                nxt = torch.where(k1[:, None], trial, nxt)
                nxt = torch.where(k2[:, None], zprev - rt * (rho / (wt * wt))[:, None], nxt)
                left = left & ~k1 & ~k2
                tau = torch.where(left, 0.5 * tau, tau)
            z = torch.where(left[:, None], tz, nxt)
        return self.T(z, x0)

    @staticmethod
    def lsq(Y, S, r):
        """S g with g the least squares solution of Y g = r, by orthogonalising Y's columns twice."""
        q, R = [], {}
        for j, y in enumerate(Y):
            v = y
            for _ in range(2):
                for i, qi in enumerate(q):
                    c = (qi * v).sum(1)
                    R[i, j] = R.get((i, j), 0) + c
                    v = v - qi * c[:, None]
            R[j, j] = v.norm(dim=1)
            q.append(v / R[j, j][:, None])
        b = [(qi * r).sum(1) for qi in q]
        g = [None] * len(Y)
        for j in range(len(Y) - 1, -1, -1):
            g[j] = (b[j] - sum(R[j, k] * g[k] for k in range(j + 1, len(Y)))) / R[j, j]
        return sum(s * c[:, None] for s, c in zip(S, g))


def _exact_network(case, seed):
    dims, params, scale, shift = _network(case, seed)
    parts, at = [], 0
    for a, b in zip(dims[:-1], dims[1:]):
        for shape in ((a, b), (b,)):
            size = int(np.prod(shape))
            parts.append(torch.tensor(params[at:at + size].reshape(shape), dtype=torch.float64, device="cuda"))
            at += size
    x = torch.tensor(_initial_states(case["problem"], seed, case["count"]), device="cuda")

    def forward(x):
        for k in range(0, len(parts) - 2, 2):
            x = torch.nn.functional.gelu(x @ parts[k] + parts[k + 1])
        return x @ parts[-2] + parts[-1]

    if case["kind"] == "predict":
        y = forward(x / 0.5)
        return y * torch.tensor(scale, device="cuda").double() + torch.tensor(shift, device="cuda").double()
    targets = _targets(case, seed, dims[-1]).double()
    mean, std = targets.mean(0), targets.std(0, unbiased=False)
    targets = (targets - mean) / std
    x = (x - x.mean(0)) / x.std(0, unbiased=False)
    losses = []
    m, v = [torch.zeros_like(p) for p in parts], [torch.zeros_like(p) for p in parts]
    for step in range(1, case["epochs"] + 1):
        for p in parts:
            p.requires_grad_(True)
        loss = (forward(x) - targets).square().mean()
        grads = torch.autograd.grad(loss, parts)
        losses.append(float(loss.detach()))
        for k, g in enumerate(grads):
            parts[k] = parts[k].detach()
            m[k].mul_(0.9).add_(0.1 * g)
            v[k].mul_(0.999).add_(0.001 * g * g)
            parts[k] -= 1e-4 * (m[k] / (1 - 0.9 ** step)) / ((v[k] / (1 - 0.999 ** step)).sqrt() + 1e-8)
    return {"loss": np.array(losses), "params": torch.cat([p.reshape(-1) for p in parts])}


def exact(case, seed):
    if case["kind"] in ("predict", "train"):
        return _exact_network(case, seed)
    names, states = _instances(case), _case_states(case, seed)
    done = [None] * len(names)
    for name in sorted(set(names)):
        plant = _Plant(name, "cuda")
        mine = [k for k, v in enumerate(names) if v == name]
        rows = _rows(case, seed, plant.n) if case.get("warm") else None
        for a in range(0, len(mine), 512):
            some = mine[a:a + 512]
            x0 = torch.tensor(np.array([states[k] for k in some]), device="cuda")
            z = torch.zeros((len(some), plant.n), dtype=torch.float64, device="cuda") if rows is None else rows[some].double()
            z = plant.solve(x0, z, rows is not None, case["method"], case["iters"])
            for k, row in zip(some, z):
                done[k] = row
    z = torch.stack(done) if case["kind"] == "shared" else torch.cat(done).cpu().numpy()
    return {"z": z, "iters": None, "status": None}
