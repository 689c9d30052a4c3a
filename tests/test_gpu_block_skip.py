"""Tile products that leave out zero 16 x 16 blocks: the Schur complement of
each subdomain against the dense elimination of its interior, on meshes whose
factor tiles are partly empty, on boxes of odd sizes (ragged last tiles), and
with couplings between arbitrary interior dofs added to the mesh pattern, so
that nonzero blocks lie where no mesh puts them.  FP64 and FP32 factors."""
import numpy as np
import pytest

import bddcml_amd
from bddcml_amd.cube import BoxProblem, CubeProblem

pytestmark = pytest.mark.gpu


def with_couplings(d, rng, n):
    """n couplings a (u_i - u_j)^2 between random dofs of the subdomain that
    are on its boundary neither of the mesh nor of a neighbour."""
    nnod = d["nnods"]
    xyz = d["xyz"]
    inside = np.ones(nnod, dtype=bool)
    for k in range(3):
        inside &= (xyz[:, k] > xyz[:, k].min()) & (xyz[:, k] < xyz[:, k].max())
    free = np.flatnonzero(np.repeat(inside, d["nndf"]))
    if len(free) < 2:
        return d
    base = int(d["i_sparse"].min())
    i, j = rng.choice(free, n), rng.choice(free, n)
    i, j = i[i != j], j[i != j]
    a = rng.uniform(0.01, 0.1, len(i)) * np.abs(d["a_sparse"]).max()
    d = dict(d)
    d["i_sparse"] = np.concatenate([d["i_sparse"], i + base, j + base, np.minimum(i, j) + base]).astype(np.int32)
    d["j_sparse"] = np.concatenate([d["j_sparse"], i + base, j + base, np.maximum(i, j) + base]).astype(np.int32)
    d["a_sparse"] = np.concatenate([d["a_sparse"], a, a, -a])
    return d


@pytest.mark.parametrize("refined", [0, 1])
@pytest.mark.parametrize("case", ["poisson 3", "poisson 10", "elasticity 6", "boxes", "coupled",
                                  "coupled elasticity"])
def test_schur_complement_equals_dense_elimination(case, refined):
    print("case block skip", case, refined, flush=True)
    p = {"poisson 3": lambda: CubeProblem(3, 2, rhs="random"),
         "poisson 10": lambda: CubeProblem(10, 2, rhs="random"),
         "elasticity 6": lambda: CubeProblem(6, 2, kind="elasticity", rhs="random"),
         "boxes": lambda: BoxProblem(17, 7, layers=4, jump=1e2),
         "coupled": lambda: CubeProblem(11, 2, rhs="random"),
         "coupled elasticity": lambda: CubeProblem(7, 2, kind="elasticity", rhs="random")}[case]()
    rng = np.random.RandomState(11)
    subs = [with_couplings(d, rng, 30 + 40 * k) if case.startswith("coupled") else d
            for k, d in enumerate(p.subdomains())]
    b = bddcml_amd.Bddcml()
    b.init(2, [p.nsub, 1], numbase=p.numbase)
    b.set_option("refinement", refined)
    for d in subs:
        b.upload_subdomain_data(d)
    b.setup_preconditioner()
    worst = 0.0
    for s, d in enumerate(subs):
        n = d["ndofs"]
        A = np.zeros((n, n))
        i, j = d["i_sparse"] - p.numbase, d["j_sparse"] - p.numbase
        np.add.at(A, (i, j), d["a_sparse"])
        np.add.at(A, (j[i != j], i[i != j]), d["a_sparse"][i != j])
        fix = d["ifix"] > 0
        g, _ = b.sub_maps(s + p.numbase)
        of = {int(v) - p.numbase: k for k, v in enumerate(d["isvgvn"])}
        ii = np.array([of[int(v)] for v in g])
        S = b.sub_matrix(s + p.numbase)
        # fixed dofs are decoupled before the elimination; rows of fixed
        # interface dofs are not compared
        io = np.setdiff1d(np.flatnonzero(~fix), ii)
        ref = A[np.ix_(ii, ii)]
        if len(io):
            ref = ref - A[np.ix_(ii, io)] @ np.linalg.solve(A[np.ix_(io, io)], A[np.ix_(io, ii)])
        k = np.flatnonzero(~fix[ii])
        err = np.abs(S - ref)[np.ix_(k, k)].max() / np.abs(ref[np.ix_(k, k)]).max()
        # elimination of n dofs: n eps growth-free for a positive definite
        # matrix (Cholesky), with eps of the factor's type
        eps = 2.0 ** -24 if refined else 2.0 ** -53
        worst = max(worst, err / (n * eps))
    b.finalize()
    assert worst <= 1.0, worst
