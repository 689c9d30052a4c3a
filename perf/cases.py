"""Timed cases of the library: what a program that solves with it has it do.

A case takes one of three paths, each through the entry points of
``bddcml_amd.Bddcml`` and ``bddcml_amd.adjoint.AdjointSolver``:

- ``solve``: a new problem, the whole call sequence of the reference's
  drivers: init, upload of every subdomain, setup, solve, download of the
  global solution, finalize.
- ``resolve``: a new right-hand side on a kept setup (time steps, load
  cases): new data of every subdomain, setup_new_data, solve, download.
- ``adjoint``: the backward direction of a differentiable solve: adjoint
  solve on the kept setup, then the gradient with respect to every element
  coefficient.

The library holds one problem per process, so the kept setup of the last two
belongs to the case (its matrix does not depend on the seed) and is made when
the process does not hold it.  The data is host data by nature: subdomain
meshes and element-assembled triplets, as the reference's interface takes
them.
"""
import math

import numpy as np
import torch

import bddcml_amd
from bddcml_amd.adjoint import AdjointSolver
from bddcml_amd.cube import BoxProblem, CubeProblem, lognormal, uniform01

DEFAULTS = dict(path="solve", mesh="cube", physics="poisson", coef="const", form="fp64", method=0,
                weights=0, nsub2=0, adaptive=0, inverse=2, layers=0, jump=1.0, tol=1e-8)


def listed():
    def case(name, **kw):
        return dict(DEFAULTS, name=name, **kw)

    return [
        # the smallest call: a few hundred dofs, all latency (a unit test, a
        # coupled code with a small subproblem)
        case("poisson 8^3", nel=4, nsub=2),
        # a medium problem with the default options
        case("poisson 64^3", nel=16, nsub=4),
        # the headline problem: 2.1 M dofs, 512 subdomains of 16^3 elements
        case("poisson 128^3", nel=16, nsub=8),
        # the form with FP32 factorizations and FP64 refinement
        case("poisson 96^3 refined", nel=16, nsub=6, form="refined"),
        # heterogeneous coefficients, odd subdomain size, FP32 preconditioner,
        # the second Krylov method, stiffness weights
        case("lognormal 65^3 bicgstab", nel=13, nsub=5, coef="lognormal", form="mixed", method=1,
             weights=1),
        # three dofs per node: wide element matrices, denser interfaces
        case("elasticity 32^3", nel=8, nsub=4, physics="elasticity"),
        # uneven subdomains with stiff layers through them, many iterations,
        # a second level in place of the dense coarse solve
        case("boxes 40^3 three levels", mesh="boxes", physics="elasticity", coef="layers", nel=40,
             nsub=36, nsub2=6, layers=9, jump=1e3, weights=1),
        # adaptive face constraints: setup dominated by the face eigenproblems
        case("boxes 24^3 adaptive", mesh="boxes", physics="elasticity", coef="layers", nel=24,
             nsub=12, layers=9, jump=1e3, weights=1, adaptive=1),
        # time stepping on the headline problem: the default options, and the
        # refined form with the inverse of the local operator asked for at
        # setup
        case("poisson 128^3 new rhs", path="resolve", nel=16, nsub=8),
        case("poisson 128^3 new rhs refined", path="resolve", nel=16, nsub=8, form="refined",
             inverse=1),
        # load cases on the uneven elasticity problem
        case("boxes 40^3 new rhs", path="resolve", mesh="boxes", physics="elasticity",
             coef="layers", nel=40, nsub=36, layers=9, jump=1e3, weights=1),
        # gradient with respect to 262,144 element coefficients
        case("adjoint gradient 64^3", path="adjoint", coef="lognormal", nel=8, nsub=8, tol=1e-10),
    ]


def draw(rng):
    """One more case: total mesh size, subdomain size, physics, coefficients,
    precision form, Krylov method and path spread over the ranges above."""
    c = dict(DEFAULTS)

    def log_int(lo, hi):
        return int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))

    c["path"] = rng.choice(["solve", "solve", "solve", "resolve", "resolve", "adjoint"])
    if c["path"] == "adjoint":
        c.update(coef="lognormal", tol=1e-10)
    else:
        c["mesh"] = rng.choice(["cube", "cube", "boxes"])
        c["physics"] = rng.choice(["poisson", "poisson", "elasticity"])
        c["form"] = rng.choice(["fp64", "fp64", "mixed", "refined"])
        if c["path"] == "resolve" and c["form"] != "fp64":
            c["inverse"] = 1
    elastic = c["physics"] == "elasticity"
    if c["mesh"] == "cube":
        c["nel"] = rng.randint(3, 9 if elastic else 17)
        edge = (36 if elastic else 110) if c["path"] != "adjoint" else 64
        c["nsub"] = log_int(2, max(2, edge // c["nel"]))
        c["method"] = rng.choice([0, 0, 0, 1]) if c["path"] != "adjoint" else 0
        if c["path"] == "solve" and rng.random() < 0.4:
            c.update(coef="lognormal", weights=rng.choice([0, 1]))
    else:
        c["nel"] = log_int(10, 36 if elastic else 72)
        sub = rng.randint(5, 11 if elastic else 17)  # mean subdomain edge
        c["nsub"] = min(400, max(4, round((c["nel"] / sub) ** 3)))
        c.update(coef="layers", layers=rng.randint(1, 9), jump=rng.choice([10.0, 100.0, 1000.0]),
                 weights=1)
        if c["nsub"] >= 24 and rng.random() < 0.4:
            c["nsub2"] = max(2, c["nsub"] // 6)
        elif (c["path"] == "solve" and c["form"] == "fp64" and c["nel"] <= 28
              and rng.random() < 0.4):
            c["adaptive"] = 1
    return c


# ------------------------------------------------------------------ inputs
_mesh = {"key": None}  # problem and subdomains of the last seed-independent matrix


def _key(case):
    return tuple(sorted((k, v) for k, v in case.items() if k != "name"))


def _problem(case, coef=None):
    if case["mesh"] == "boxes":
        return BoxProblem(case["nel"], case["nsub"], seed=3, kind=case["physics"],
                          layers=case["layers"], jump=case["jump"], rhs="const")
    return CubeProblem(case["nel"], case["nsub"], kind=case["physics"], rhs="const",
                       coef=None if coef is None else lambda e: coef[e])


def _coefficients(case, seed):
    """Log-normal element coefficients (mu 0, sigma 1), or None."""
    if case["coef"] != "lognormal":
        return None
    return lognormal(seed, np.arange((case["nel"] * case["nsub"]) ** 3))


def _subdomains(case, seed):
    """The problem and its subdomains for the path "solve" or "resolve": the
    right-hand side (uniform in [-1, 1], zero at fixed dofs) and log-normal
    coefficients come from the seed, the rest from the case."""
    if case["coef"] == "lognormal":
        p = _problem(case, _coefficients(case, seed))
        subs = list(p.subdomains())
    else:
        key = _key({k: case[k] for k in ("mesh", "physics", "nel", "nsub", "layers", "jump")})
        if _mesh["key"] != key:
            p = _problem(case)
            _mesh.update(key=key, p=p, subs=list(p.subdomains()))
        p, subs = _mesh["p"], _mesh["subs"]
    value = 2.0 * uniform01(seed, np.arange(p.ndof)) - 1.0
    out = []
    for d in subs:
        rhs = value[d["isvgvn"] - p.numbase]
        rhs[d["ifix"] > 0] = 0.0
        out.append(dict(d, rhs=rhs))
    return p, out


# ------------------------------------------------------------------- paths
_held = {"key": None}  # the case whose setup the library holds, and its handle


def _upload_and_setup(case, p, subs):
    _held["key"] = None
    b = bddcml_amd.Bddcml()
    nsublev = [p.nsub] + ([case["nsub2"]] if case["nsub2"] else []) + [1]
    b.init(len(nsublev), nsublev, numbase=p.numbase)
    if case["form"] == "mixed":
        b.set_option("precision", 32)
    elif case["form"] == "refined":
        b.set_option("refinement", 1)
    b.set_option("explicit_inverse", case["inverse"])
    for d in subs:
        b.upload_subdomain_data(d)
    b.setup_preconditioner(1, 0, 1, 1, 1, case["adaptive"], 0, case["weights"])
    return b


def _solve(case, b, p):
    _, reason, _ = b.solve(case["method"], case["tol"], 2000, 200)
    if reason != 0:
        raise RuntimeError(f"not converged: reason {reason}")
    return b.download_global_solution(p.ndof)


def _hold(case, state):
    """The kept setup of the case's matrix (made again if the process has
    gone on to another problem since)."""
    key = _key(case)
    if _held["key"] != key:
        if case["path"] == "adjoint":
            k = _coefficients(case, 5)
            sol = AdjointSolver(lambda kk: CubeProblem(case["nel"], case["nsub"], rhs="random",
                                                       seed=5, coef=lambda e: kk[e]),
                                _problem(case).kref, tol=case["tol"])
            _held["key"] = None
            u = sol.forward(k)
            _held.update(key=key, handle=sol, u=u)
        else:
            b = _upload_and_setup(case, state["p"], state["subs"])
            _held.update(key=key, handle=b, u=None)
    return _held["handle"]


def prepare(case, seed):
    case = dict(DEFAULTS, **case)
    state = {"case": case}
    if case["path"] == "adjoint":
        p = _problem(case)
        state.update(p=p, dJdu=2.0 * uniform01(seed, np.arange(p.ndof)) - 1.0)
    else:
        p, subs = _subdomains(case, seed)
        state.update(p=p, subs=subs)
    if case["path"] != "solve":
        _hold(case, state)
    return state


def run(state):
    case, p = state["case"], state["p"]
    if case["path"] == "solve":
        b = _upload_and_setup(case, p, state["subs"])
        u = _solve(case, b, p)
        b.finalize()
        return {"u": u}
    handle = _hold(case, state)
    if case["path"] == "resolve":
        for d in state["subs"]:
            handle.change_subdomain_data(d)
        handle.setup_new_data()
        return {"u": _solve(case, handle, p)}
    lam = handle.adjoint(state["dJdu"])
    return {"lam": lam, "grad": handle.gradient(_held["u"], lam)}


# ----------------------------------------------------- counts and checking
def _sizes(case):
    """dofs, element-matrix triplets, mean interface dofs of a subdomain."""
    ndf = 3 if case["physics"] == "elasticity" else 1
    edge = case["nel"] * case["nsub"] if case["mesh"] == "cube" else case["nel"]
    nsub = case["nsub"] ** 3 if case["mesh"] == "cube" else case["nsub"]
    ne = 8 * ndf
    m = edge / nsub ** (1.0 / 3.0) + 1  # nodes along a subdomain edge
    share = 1.0 - nsub ** (-1.0 / 3.0)  # faces that are not on the boundary
    ni = ndf * share * (m ** 3 - max(m - 2, 0) ** 3)
    return (edge + 1) ** 3 * ndf, edge ** 3 * ne * (ne + 1) // 2, ni, nsub


def work(case):
    """Host data in and the solution out once, and, per iteration of a
    nominal ten, one read of a symmetric interface operator (half of it
    stored) for the operator and one for its preconditioner; for a new
    problem the Cholesky factorization of a dense interface matrix per
    subdomain."""
    case = dict(DEFAULTS, **case)
    ndof, ntrip, ni, nsub = _sizes(case)
    applies = 10 * 2
    op_flops = applies * nsub * 2.0 * ni * ni
    if case["path"] == "solve":
        return {"bytes": 16.0 * ntrip + 60.0 * ndof,
                "flops": op_flops + nsub * ni ** 3 / 3.0}
    size = 8.0 if case["form"] == "fp64" else 4.0
    return {"bytes": 40.0 * ndof + applies * nsub * ni * ni / 2.0 * size, "flops": op_flops}


def tolerance(case):
    """Solutions of the same stopping test: a relative residual of 1e-8 left
    errors up to 9.7e-9 against exact() over these ranges, 1e-10 (adjoint)
    up to 3.1e-11; four times that, as an iteration more or fewer shifts
    them."""
    return {"rel": 1.2e-10} if dict(DEFAULTS, **case)["path"] == "adjoint" else {"rel": 4e-8}


def _ell(p, subs):
    """The assembled global matrix with eliminated Dirichlet rows as padded
    rows (columns, values), and the fixed dofs, on the GPU."""
    dev = "cuda" if torch.cuda.is_available() else "cpu"
    n, b = p.ndof, p.numbase
    key, val = None, None

    def summed(key, val):
        key, inv = torch.unique(key, return_inverse=True)
        return key, torch.zeros(key.numel(), dtype=torch.float64, device=dev).index_add_(0, inv, val)

    fixed = torch.zeros(n, dtype=torch.bool, device=dev)
    batch = []
    for s, d in enumerate(subs):
        g = torch.from_numpy(d["isvgvn"].astype(np.int64) - b).to(dev)
        i = g[torch.from_numpy(d["i_sparse"].astype(np.int64) - b).to(dev)]
        j = g[torch.from_numpy(d["j_sparse"].astype(np.int64) - b).to(dev)]
        a = torch.from_numpy(np.asarray(d["a_sparse"], dtype=np.float64)).to(dev)
        off = i != j
        batch.append(summed(torch.cat([i * n + j, (j * n + i)[off]]), torch.cat([a, a[off]])))
        fixed[g[torch.from_numpy(d["ifix"] > 0).to(dev)]] = True
        if len(batch) == 64 or s + 1 == len(subs):
            if key is not None:
                batch.append((key, val))
            key, val = summed(torch.cat([k for k, _ in batch]), torch.cat([v for _, v in batch]))
            batch = []
    row, col = key // n, key % n
    keep = (row == col) | ~(fixed[row] | fixed[col])
    row, col, val = row[keep], col[keep], val[keep]
    count = torch.bincount(row, minlength=n)
    start = torch.cumsum(count, 0) - count
    slot = torch.arange(row.numel(), device=dev) - start[row]
    width = int(count.max())
    cols = torch.zeros(n, width, dtype=torch.int64, device=dev)
    vals = torch.zeros(n, width, dtype=torch.float64, device=dev)
    cols[row, slot] = col
    vals[row, slot] = val
    diag = torch.zeros(n, dtype=torch.float64, device=dev)
    diag[row[row == col]] = val[row == col]
    return cols, vals, diag, fixed


def _cg(cols, vals, diag, f, tol=1e-14, maxit=40000):
    """Conjugate gradients with the diagonal as preconditioner, FP64."""
    u = torch.zeros_like(f)
    r = f.clone()
    z = r / diag
    p = z.clone()
    rz = (r * z).sum()
    stop = tol * float(torch.linalg.vector_norm(f))
    for it in range(maxit):
        ap = (vals * p[cols]).sum(1)
        alpha = rz / (p * ap).sum()
        u += alpha * p
        r -= alpha * ap
        z = r / diag
        new = (r * z).sum()
        p = z + (new / rz) * p
        rz = new
        if it % 50 == 49 and float(torch.linalg.vector_norm(r)) <= stop:
            return u
    return None


def exact(case, seed):
    """The solution of the assembled system by conjugate gradients in FP64
    to a residual of 1e-14, and the element gradient from it, in plain
    torch."""
    case = dict(DEFAULTS, **case)
    if case["path"] == "adjoint":
        k = _coefficients(case, 5)
        p = _problem(case, k)
        subs = list(p.subdomains())
        f0 = np.zeros(p.ndof)
        f0[:] = 2.0 * uniform01(5, np.arange(p.ndof)) - 1.0
        dJdu = 2.0 * uniform01(seed, np.arange(p.ndof)) - 1.0
        cols, vals, diag, fixed = _ell(p, subs)
        sols = []
        for rhs in (f0, dJdu):
            f = torch.from_numpy(rhs).to(diag.device)
            f[fixed] = 0.0
            sols.append(_cg(cols, vals, diag, f))
        if sols[0] is None or sols[1] is None:
            return None
        u, lam = (x.cpu().numpy() for x in sols)
        grad = np.zeros(p.nelem)
        for d in subs:
            dof = (d["isvgvn"] - p.numbase)[d["inet"].reshape(-1, 8) - p.numbase]
            grad[d["isegn"] - p.numbase] = -np.einsum("ei,ij,ej->e", lam[dof], p.kref, u[dof])
        return {"lam": lam, "grad": grad}
    p, subs = _subdomains(case, seed)
    cols, vals, diag, fixed = _ell(p, subs)
    f = torch.zeros(p.ndof, dtype=torch.float64, device=diag.device)
    for d in subs:
        f[torch.from_numpy(d["isvgvn"].astype(np.int64) - p.numbase).to(f.device)] = (
            torch.from_numpy(d["rhs"]).to(f.device))
    u = _cg(cols, vals, diag, f)
    return None if u is None else {"u": u.cpu().numpy()}
