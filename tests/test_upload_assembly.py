"""Triplet assembly of bddcml_upload_subdomain_data_c at sizes where one and
several host threads share it: any input order gives the same matrix, and a
bad entry is refused with its message wherever it stands."""
import numpy as np
import pytest

import bddcml_amd
from bddcml_amd.cube import CubeProblem


def _shuffled(d, seed, full=False):
    rng = np.random.RandomState(seed)
    i, j, a = d["i_sparse"], d["j_sparse"], d["a_sparse"]
    if full:  # both triangles
        off = i != j
        i, j, a = (np.concatenate([i, j[off]]), np.concatenate([j, i[off]]),
                   np.concatenate([a, a[off]]))
    o = rng.permutation(len(a))
    return dict(d, i_sparse=i[o].copy(), j_sparse=j[o].copy(), a_sparse=a[o].copy(),
                matrixtype=0 if full else d["matrixtype"])


# 2,304 triplets: one thread; 18,432 and 62,208: two and seven shares;
# elasticity rows of up to 648 triplets (the long-row sort)
@pytest.mark.gpu
@pytest.mark.parametrize("nel,kind,full", [(4, "poisson", False), (8, "poisson", False),
                                           (12, "poisson", True), (6, "elasticity", False)])
def test_input_order_does_not_matter(nel, kind, full):
    print("case upload order", nel, kind, full, flush=True)
    p = CubeProblem(nel, 2, kind=kind, rhs="random", seed=3)
    mats = []
    for shuffle in (False, True):
        b = bddcml_amd.Bddcml()
        b.init(2, [p.nsub, 1], numbase=p.numbase)
        for k, d in enumerate(p.subdomains()):
            b.upload_subdomain_data(_shuffled(d, k, full) if shuffle else d)
        b.setup_preconditioner(0 if full and shuffle else 1)
        mats.append([b.sub_matrix(s + p.numbase) for s in range(p.nsub)])
        b.finalize()
    for x, y in zip(*mats):
        # the entries' sums differ by reordered additions of 8 terms at most
        assert np.abs(x - y).max() <= 1e-12 * np.abs(x).max()


@pytest.mark.parametrize("nel", [4, 12])
@pytest.mark.parametrize("place", [0, 0.4, 1.0])
def test_bad_entries_are_refused(nel, place):
    p = CubeProblem(nel, 2)
    d = p.subdomain(0)
    k = int(place * (len(d["a_sparse"]) - 1))
    for i, j, text in ((5, 3, "upper triangle"), (1, d["ndofs"] + 1, "out of range"),
                       (0, 3, "out of range")):
        bad = dict(d, i_sparse=d["i_sparse"].copy(), j_sparse=d["j_sparse"].copy())
        bad["i_sparse"][k], bad["j_sparse"][k] = i, j
        b = bddcml_amd.Bddcml()
        b.init(2, [p.nsub, 1], numbase=p.numbase)
        b.set_option("plan_only", 1)
        with pytest.raises(RuntimeError, match=text):
            b.upload_subdomain_data(bad)
        b.upload_subdomain_data(d)
        b.finalize()


def test_first_bad_entry_names_the_error():
    """Two bad entries in different threads' shares: the first one counts."""
    p = CubeProblem(12, 2)
    d = p.subdomain(0)
    n = len(d["a_sparse"])
    bad = dict(d, i_sparse=d["i_sparse"].copy(), j_sparse=d["j_sparse"].copy())
    bad["i_sparse"][n // 3], bad["j_sparse"][n // 3] = 9, 2
    bad["j_sparse"][n - 1] = d["ndofs"] + 7
    b = bddcml_amd.Bddcml()
    b.init(2, [p.nsub, 1], numbase=p.numbase)
    b.set_option("plan_only", 1)
    with pytest.raises(RuntimeError, match="upper triangle"):
        b.upload_subdomain_data(bad)
    b.finalize()
