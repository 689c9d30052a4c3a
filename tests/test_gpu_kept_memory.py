"""Device memory kept between problems: reused by the next problem with the
same results, given back when a whole problem did not use it, and given back
entirely by a finalize without a problem."""
import ctypes as C

import numpy as np
import pytest

import bddcml_amd
from bddcml_amd.cube import CubeProblem

pytestmark = pytest.mark.gpu


def _free():
    # of the HIP runtime the library is linked with
    free, total = C.c_size_t(), C.c_size_t()
    assert bddcml_amd.lib().hipMemGetInfo(C.byref(free), C.byref(total)) == 0
    return free.value


def _solve(nel, ns, kind="poisson"):
    p = CubeProblem(nel, ns, kind=kind, rhs="random", seed=3)
    b, (it, reason, _) = bddcml_amd.solve_cube(p, tol=1e-9)
    assert reason == 0
    u = b.interface_solution()
    b.finalize()
    return it, u


def test_memory_is_reused_and_given_back():
    print("case kept memory", flush=True)
    empty = bddcml_amd.Bddcml()
    _solve(16, 2)  # the runtime's own memory is there after a first solve
    empty.finalize()
    start = _free()
    first = _solve(16, 2)  # some 200 MB
    kept = start - _free()
    assert kept > 100 << 20
    again = _solve(16, 2)
    assert start - _free() <= kept + (16 << 20)
    assert first[0] == again[0] and np.array_equal(first[1], again[1])
    # problems of other sizes in between change nothing
    small = _solve(4, 2)
    _solve(5, 2, kind="elasticity")
    assert start - _free() < kept // 2  # the large blocks went unused and back
    other = _solve(4, 2)
    assert small[0] == other[0] and np.array_equal(small[1], other[1])
    assert np.array_equal(_solve(16, 2)[1], first[1])
    empty.finalize()
    assert start - _free() < 16 << 20
