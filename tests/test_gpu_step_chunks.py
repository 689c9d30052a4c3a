"""Factorizations and sweeps whose steps are cut into chunks (few subdomains:
every sequence of more than four tile rows): the coarse basis against its
energies, and the local corrections by the inverse built in chunks against
those by sweeps over the factor, for 1 to 16 tile rows, subdomains of mixed
sizes, FP64 and FP32 factors."""
import numpy as np
import pytest

import bddcml_amd
from bddcml_amd.cube import BoxProblem, CubeProblem

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("precision", [64, 32])
@pytest.mark.parametrize("case", ["poisson 3", "poisson 8", "poisson 9", "poisson 10", "poisson 14",
                                  "elasticity 10", "boxes"])
def test_chunked_factor_and_inverse(case, precision):
    print("case step chunks", case, precision, flush=True)
    if case == "boxes":
        p = BoxProblem(19, 7, layers=4, jump=1e2)
    else:
        kind, nel = case.split()
        p = CubeProblem(int(nel), 2, kind=kind, rhs="random", seed=4)
    # FP64 values in the basis energies; the factor's type in the applies
    eps = 2.0 ** (-53 if precision == 64 else -24)
    out = []
    for inverse in (0, 1):
        b = bddcml_amd.Bddcml()
        b.init(2, [p.nsub, 1], numbase=p.numbase)
        b.set_option("precision", precision)
        b.set_option("explicit_inverse", inverse)
        for d in p.subdomains():
            b.upload_subdomain_data(d)
        b.setup_preconditioner()
        for s in range(p.nsub):
            S = b.sub_matrix(s + p.numbase)
            phi, ac = b.sub_coarse(s + p.numbase)
            n = len(S)
            scale = np.linalg.norm(phi.T) ** 2 * np.abs(S).max()
            assert np.abs(phi.T @ S @ phi - ac).max() <= 8 * n * eps * scale
        x = np.random.RandomState(6).uniform(-1, 1, len(b.interface_dofs()))
        out.append(b.apply_pc(x))
        b.finalize()
    # two backward stable applies of one matrix of condition <= 1e4
    assert np.abs(out[0] - out[1]).max() <= 1e4 * eps * np.abs(out[0]).max()
