"""The sweeps over interior and interface factors in the forms that the number
of subdomains selects (up to 256, up to 1023 and more), FP64 and FP32 factors:
the residual of the assembled matrix at the solution, which the sweeps of the
reduced right-hand side and of the interiors leave at the tolerance of the
interface problem."""
import numpy as np
import pytest

import bddcml_amd
from bddcml_amd.cube import CubeProblem

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("refined", [0, 1])
@pytest.mark.parametrize("nel,ns", [(9, 2), (4, 6), (4, 7), (2, 10), (2, 11)])
def test_sweeps_solve_the_interiors(nel, ns, refined):
    print("case sweep forms", nel, ns, refined, flush=True)
    p = CubeProblem(nel, ns, rhs="random", seed=8)
    b, (it, reason, _) = bddcml_amd.solve_cube(p, tol=1e-12, options={"refinement": refined})
    assert reason == 0
    u = b.download_global_solution(p.ndof)
    b.finalize()
    # the residual of the assembled matrix on the free dofs: backward stable
    # interior solves leave it at the tolerance of the interface problem
    import scipy.sparse as sp
    rows, cols, vals, f, fixed = [], [], [], np.zeros(p.ndof), np.zeros(p.ndof, dtype=bool)
    for d in p.subdomains():
        g = d["isvgvn"] - p.numbase
        i, j, a = g[d["i_sparse"] - p.numbase], g[d["j_sparse"] - p.numbase], d["a_sparse"]
        off = d["i_sparse"] != d["j_sparse"]
        rows += [i, j[off]]
        cols += [j, i[off]]
        vals += [a, a[off]]
        f[g] = d["rhs"]
        fixed[g[d["ifix"] > 0]] = True
    A = sp.csr_matrix((np.concatenate(vals), (np.concatenate(rows), np.concatenate(cols))),
                      shape=(p.ndof, p.ndof))
    r = (f - A @ u)[~fixed]
    assert np.abs(r).max() <= 1e-10 * np.abs(f).max()
