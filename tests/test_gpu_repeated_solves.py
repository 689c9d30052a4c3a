"""Many new right-hand sides on one setup: the preconditioner passes from the
sweeps to the explicit inverse between two solves (explicit_inverse = 2), and
the captured PCG iteration has to follow it in every precision form."""
import numpy as np
import pytest

import bddcml_amd
from bddcml_amd.cube import CubeProblem

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("form", [{}, {"precision": 32}, {"refinement": 1}])
@pytest.mark.parametrize("kind", ["poisson", "elasticity"])
def test_iterations_do_not_change_over_many_solves(form, kind):
    print("case repeated solves", form, kind, flush=True)
    p = CubeProblem(4, 3, kind=kind, rhs="random", seed=3)
    subs = list(p.subdomains())
    # the automatic mode against the inverse formed at setup (1) and never (0)
    runs = {}
    for mode in (0, 1, 2):
        b, (it, reason, _) = bddcml_amd.solve_cube(p, tol=1e-9, maxit=300,
                                                   options=dict(form, explicit_inverse=mode))
        out = [(it, reason, b.interface_solution())]
        for _ in range(9):
            for d in subs:
                b.change_subdomain_data(d)
            b.setup_new_data()
            it, reason, _ = b.solve(0, 1e-9, 300, 50)
            out.append((it, reason, b.interface_solution()))
        b.finalize()
        runs[mode] = out
    ref = runs[0][0]
    scale = np.abs(ref[2]).max()
    for mode, out in runs.items():
        for k, (it, reason, u) in enumerate(out):
            assert reason == 0 and abs(it - ref[0]) <= 1, (mode, k, it, reason)
            # two solutions of the same stopping test (1e-9, condition below 10)
            assert np.abs(u - ref[2]).max() < 1e-7 * scale
