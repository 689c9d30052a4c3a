"""Host work that the device waits for in a setup of many different
subdomains (one class of task lists each): the time of the interior
factorization beside that of its product launches."""
import pytest

import bddcml_amd
from bddcml_amd.cube import BoxProblem

pytestmark = pytest.mark.gpu


def test_factorization_does_not_wait_for_counts():
    print("case setup gaps", flush=True)
    p = BoxProblem(64, 120, seed=3, layers=9, jump=1e3)
    subs = list(p.subdomains())
    best = None
    for _ in range(4):
        b = bddcml_amd.Bddcml()
        b.init(2, [p.nsub, 1], numbase=p.numbase)
        for d in subs:
            b.upload_subdomain_data(d)
        b.setup_preconditioner(weights_type=1)
        t = b.timings()
        b.finalize()
        assert t["interior_flops"] > t["schur_flops"] > 0 and t["gemm_flops"] > 0
        gap = (t["ev_interior_ms"] - t["ev_gemm_ms"]) / t["ev_gemm_ms"]
        best = gap if best is None else min(best, gap)
    # tile factorizations, clearing and scattering of the tiles and the host's
    # task lists: 1.2 times the products (18.7 ms of 40.6), 2.3 times while one
    # thread counted the products' blocks before the first launch
    assert best < 1.7, best
