"""The inverses of the subdomains' constraint matrices G (kernels k_ginv with
the matrix in registers, by size class, and k_ginv_large) on the device
against numpy: the ends of every class, sizes mixed in one launch, subdomains
without constraints, a pivot that is not positive."""
import numpy as np
import pytest

import bddcml_amd

pytestmark = pytest.mark.gpu


def _spd(n, seed, scaled):
    rng = np.random.default_rng(seed)
    q = np.linalg.qr(rng.standard_normal((n, n)))[0]
    a = (q * np.logspace(0, -3, n)) @ q.T
    if scaled:  # coefficient jumps
        d = 10.0 ** rng.uniform(-2, 2, n)
        a = d[:, None] * a * d
    return (a + a.T) / 2


# the largest of a launch chooses the kernel: 32 rows a class up to 192
@pytest.mark.parametrize("sizes", [[1], [31, 2], [32, 0, 5], [33], [64, 32], [65], [96, 1], [97], [128],
                                   [129, 64], [160, 0, 159], [161], [192, 33], [193, 0, 1], [256, 192],
                                   [700], [1024, 3]])
@pytest.mark.parametrize("scaled", [False, True])
def test_inverse(sizes, scaled):
    print("case inverse", sizes, scaled, flush=True)
    mats = [_spd(n, 7 + n, scaled) if n else np.zeros((0, 0)) for n in sizes]
    out, err = bddcml_amd.selftest_inverse(mats)
    assert err == 0
    for a, x in zip(mats, out):
        n = len(a)
        if n == 0:
            continue
        # Gauss-Jordan on a positive definite matrix: n eps cond(a), and the
        # diagonal scaling of a does not enter (the steps commute with it)
        d = np.sqrt(np.diag(a))
        a, x = a / np.outer(d, d), x * np.outer(d, d)
        tol = 4 * n * np.finfo(float).eps * np.linalg.cond(a)
        assert np.linalg.norm(a @ x - np.eye(n), 2) <= tol
        assert np.linalg.norm(x - x.T, 2) <= tol * np.linalg.norm(x, 2)


@pytest.mark.parametrize("n", [20, 192, 200])
def test_a_pivot_that_is_not_positive(n):
    print("case pivot", n, flush=True)
    good, bad = _spd(n, 1, False), _spd(n, 2, False)
    bad[n // 2, n // 2] = -1.0
    out, err = bddcml_amd.selftest_inverse([good, bad])
    assert err != 0
    assert np.linalg.norm(good @ out[0] - np.eye(n), 2) <= 4 * n * 2.2e-16 * 1e3
