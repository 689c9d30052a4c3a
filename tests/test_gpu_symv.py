"""The symmetric tile GEMV against dense products with the subdomains' Schur
complements, in each form its launch can take: single-column groups (few
subdomains), grouped columns with the input in LDS (many), grouped columns
with the input gathered tile by tile (interfaces of more than 72 tiles); FP64
and FP32 tiles."""
import numpy as np
import pytest

import bddcml_amd
from bddcml_amd.cube import CubeProblem

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("refined", [0, 1])
@pytest.mark.parametrize("nel,ns,kind", [(2, 2, "poisson"), (8, 4, "poisson"), (8, 6, "poisson"),
                                         (5, 5, "elasticity"), (16, 3, "elasticity")])
def test_schur_apply_equals_dense_products(nel, ns, kind, refined):
    print("case symmetric GEMV", nel, ns, kind, refined, flush=True)
    p = CubeProblem(nel, ns, kind=kind, rhs="random", seed=3)
    b = bddcml_amd.Bddcml()
    b.init(2, [p.nsub, 1], numbase=p.numbase)
    b.set_option("refinement", refined)
    for d in p.subdomains():
        b.upload_subdomain_data(d)
    b.setup_preconditioner()
    ig = b.interface_dofs()
    pos = -np.ones(p.ndof, dtype=int)
    pos[ig] = np.arange(len(ig))
    x = np.random.RandomState(5).uniform(-1, 1, len(ig))
    y = b.apply_schur(x)
    ref = np.zeros_like(x)
    for s in range(p.nsub):
        g, _ = b.sub_maps(s + p.numbase)
        k = pos[g]
        np.add.at(ref, k, b.sub_matrix(s + p.numbase) @ x[k])
    b.finalize()
    # the same products summed in another order: n eps of the row sums of moduli
    assert np.abs(y - ref).max() <= 1e-12 * np.abs(ref).max()


@pytest.mark.parametrize("precision", [64, 32])
def test_inverse_apply_of_gathered_inputs(precision):
    """The local preconditioner through the explicit inverse, whose weighted
    input is gathered tile by tile (interfaces of up to 73 tiles), against the
    sweeps over the factor."""
    print("case gathered inverse", precision, flush=True)
    p = CubeProblem(16, 3, kind="elasticity", rhs="random", seed=3)
    subs = list(p.subdomains())
    out = []
    for inverse in (0, 1):
        b = bddcml_amd.Bddcml()
        b.init(2, [p.nsub, 1], numbase=p.numbase)
        b.set_option("precision", precision)
        b.set_option("explicit_inverse", inverse)
        for d in subs:
            b.upload_subdomain_data(d)
        b.setup_preconditioner()
        x = np.random.RandomState(6).uniform(-1, 1, len(b.interface_dofs()))
        out.append(b.apply_pc(x))
        b.finalize()
    # two backward stable applies of one matrix of condition <= 1e4
    eps = 2.0 ** (-53 if precision == 64 else -24)
    assert np.abs(out[0] - out[1]).max() <= 1e4 * eps * np.abs(out[0]).max()
