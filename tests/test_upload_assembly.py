"""Triplet assembly of bddcml_upload_subdomain_data_c, on the host (small
subdomains, full storage) and on the device (from 16,384 triplets): any input
order gives the same matrix, and a bad entry is refused with its message
wherever it stands."""
import time

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


# 2,304 triplets: one host thread; 18,432: device; 62,208 in full storage:
# several host threads; elasticity: device, rows of up to 192 triplets
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


def _matrices(p, change, matrixtype=1):
    b = bddcml_amd.Bddcml()
    b.init(2, [p.nsub, 1], numbase=p.numbase)
    for k, d in enumerate(p.subdomains()):
        b.upload_subdomain_data(change(d, k))
    b.setup_preconditioner(matrixtype)
    it, reason, _ = b.solve(0, 1e-10, 200, 50)
    assert reason == 0
    out = [b.sub_matrix(s + p.numbase) for s in range(p.nsub)], b.download_global_solution(p.ndof)
    b.finalize()
    return out


@pytest.mark.gpu
def test_long_rows_on_the_device():
    """Every triplet in 20 parts: rows of up to 1,280 entries, beyond what a
    wave of the device sort holds in LDS (512)."""
    print("case long rows", flush=True)
    p = CubeProblem(4, 2, rhs="random", seed=3)  # 46,080 triplets

    def parts(d, k):
        o = np.random.RandomState(k).permutation(20 * len(d["a_sparse"]))
        rep = lambda x: np.tile(x, 20)[o].copy()
        return dict(d, i_sparse=rep(d["i_sparse"]), j_sparse=rep(d["j_sparse"]),
                    a_sparse=rep(d["a_sparse"] / 20.0))

    (x, u), (y, v) = _matrices(p, lambda d, k: d), _matrices(p, parts)
    for a, b in zip(x, y):
        # sums of 160 terms in another order: 160 eps of the entries' sum of moduli
        assert np.abs(a - b).max() <= 1e-12 * np.abs(a).max()
    assert np.abs(u - v).max() <= 1e-9 * np.abs(u).max()


def _with_long_row(p, d, length, columns):
    """d with `length` more entries in one row, over `columns` columns in
    random order, and the diagonal that keeps the matrix positive definite."""
    rng = np.random.RandomState(length)
    n = d["ndofs"]
    r = n - 1 - columns
    v = rng.rand(length) - 0.5
    j = rng.permutation(np.arange(length) % columns) + r + 1
    add = np.bincount(j, np.abs(v), minlength=n)
    add[r] += np.abs(v).sum()
    k = np.nonzero(add)[0]
    cat = lambda x, *y: np.concatenate((x,) + y).astype(x.dtype)
    return dict(d, i_sparse=cat(d["i_sparse"], np.full(length, r) + p.numbase, k + p.numbase),
                j_sparse=cat(d["j_sparse"], j + p.numbase, k + p.numbase),
                a_sparse=cat(d["a_sparse"], v, add[k]))


# rows about the ends of what a wave (512) and a run (1,024) hold, of an even
# and an odd number of merges; one column (all duplicates) to 700
@pytest.mark.gpu
@pytest.mark.parametrize("length,columns", [(480, 400), (512, 512), (513, 512), (1024, 700), (1025, 1),
                                            (2048, 700), (2049, 700), (4097, 37), (20000, 700),
                                            (20000, 1), (70000, 2)])
def test_one_long_row(length, columns):
    """One row of many entries, of many duplicates: the device assembly
    against the host's of the same matrix in full storage."""
    print("case one long row", length, columns, flush=True)
    p = CubeProblem(8, 2, rhs="random", seed=3)
    out = []
    for full in (False, True):
        def change(d, k):
            d = _with_long_row(p, d, length, columns) if k == 0 else d
            return _shuffled(d, k, True) if full else d
        out.append(_matrices(p, change, 0 if full else 1))
    (x, u), (y, v) = out
    for a, b in zip(x, y):
        # sums of up to 70,000 terms in another order: 70,000 eps of the sum of
        # moduli, which the diagonals hold
        assert np.abs(a - b).max() <= 2e-11 * np.abs(a).max()
    assert np.abs(u - v).max() <= 1e-8 * np.abs(u).max()


@pytest.mark.gpu
@pytest.mark.parametrize("columns", [1, 364])
def test_a_long_row_costs_no_more_than_its_entries(columns):
    """20,000 more entries in one row: as the same number spread over all rows,
    and 50 ms (ranks over the whole row took 590 ms)."""
    print("case cost of a long row", columns, flush=True)
    p = CubeProblem(8, 2, rhs="random", seed=3)
    subs = list(p.subdomains())
    d0 = subs[0]
    n = d0["ndofs"]
    zeros = np.zeros(20000)
    lo = np.random.RandomState(1).randint(0, n, (2, 20000))
    best = []
    for i, j in ((lo.min(0), lo.max(0)),
                 (np.full(20000, n - 1 - columns), n - columns + np.arange(20000) % columns)):
        d = dict(d0, i_sparse=np.concatenate([d0["i_sparse"], i + p.numbase]).astype(np.int32),
                 j_sparse=np.concatenate([d0["j_sparse"], j + p.numbase]).astype(np.int32),
                 a_sparse=np.concatenate([d0["a_sparse"], zeros]))
        t = []
        for _ in range(3):
            b = bddcml_amd.Bddcml()
            b.init(2, [p.nsub, 1], numbase=p.numbase)
            t0 = time.perf_counter()
            for s in [d] + subs[1:]:
                b.upload_subdomain_data(s)
            b.setup_preconditioner()
            t.append(time.perf_counter() - t0)
            b.finalize()
        best.append(min(t))
    assert best[1] < best[0] + 0.05, best


@pytest.mark.gpu
def test_room_for_the_assembled_entries_only():
    """9.4 M triplets of 151 MB, 4.3 M assembled entries of 69 MB: the device
    assembly, in several batches, holds no more than the assembled entries,
    which are all that the host assembly (full storage) sends, row starts and
    flags."""
    print("case room for entries", flush=True)
    p = CubeProblem(16, 4, rhs="random", seed=3)
    held = []
    for full in (True, False):
        b = bddcml_amd.Bddcml()
        b.init(2, [p.nsub, 1], numbase=p.numbase)
        for k, d in enumerate(p.subdomains()):
            b.upload_subdomain_data(_shuffled(d, k, True) if full else d)
        b.setup_preconditioner(0 if full else 1)
        held.append(b.device_memory()[0])
        assert b.solve(0, 1e-8, 100, 50)[1] == 0
        b.finalize()
    assert b.device_memory()[0] == 0.0
    # 13 to 25 bytes a dof beside the entries, blocks of up to 32 MiB (with room
    # for all triplets 192 MB more)
    assert held[1] <= held[0] + 42e6, held


@pytest.mark.gpu
@pytest.mark.parametrize("nel", [4, 8, 9])
def test_fixed_dofs_without_diagonal(nel):
    """Missing diagonals of fixed dofs become 1, nonzero fixed values move to
    the right-hand side: device assembly against the host's full storage."""
    print("case missing diagonals", nel, flush=True)
    p = CubeProblem(nel, 2, rhs="random", seed=3, dirichlet="random")

    def drop(d, k):
        b = p.numbase
        keep = (d["i_sparse"] != d["j_sparse"]) | (d["ifix"][d["i_sparse"] - b] == 0)
        return dict(d, **{n: d[n][keep].copy() for n in ("i_sparse", "j_sparse", "a_sparse")})

    (x, u) = _matrices(p, drop)
    (y, v) = _matrices(p, lambda d, k: _shuffled(drop(d, k), k, full=True), matrixtype=0)
    for a, b in zip(x, y):
        assert np.abs(a - b).max() <= 1e-12 * np.abs(a).max()
    assert np.abs(u - v).max() <= 1e-8 * np.abs(u).max()
    # fixed values come back as given
    for d in p.subdomains():
        g = d["isvgvn"][d["ifix"] > 0] - p.numbase
        assert np.allclose(u[g], d["fixv"][d["ifix"] > 0], rtol=1e-12, atol=0)


@pytest.mark.gpu
@pytest.mark.parametrize("kind", ["poisson", "elasticity"])
def test_stiffness_weights_and_reactions(kind):
    """The diagonal and the Dirichlet couplings read back from the device
    assembly: stiffness weights and reactions against the host's assembly of
    the same matrix in full storage."""
    print("case weights, reactions", kind, flush=True)
    n = 6 if kind == "elasticity" else 9
    p = CubeProblem(n, 2, kind=kind, rhs="random", seed=3, dirichlet="random",
                    coef=lambda e: 1.0 + (e % 7))
    out = []
    for full in (False, True):
        b = bddcml_amd.Bddcml()
        b.init(2, [p.nsub, 1], numbase=p.numbase)
        for k, d in enumerate(p.subdomains()):
            b.upload_subdomain_data(_shuffled(d, k, True) if full else d)
        b.setup_preconditioner(0 if full else 1, weights_type=1)
        it, reason, _ = b.solve(0, 1e-11, 200, 50)
        assert reason == 0
        r = np.random.RandomState(1).rand(b.counts()["nig"])
        out.append((it, b.apply_pc(r), b.download_global_solution(p.ndof),
                    b.download_global_reactions(p.ndof)))
        b.finalize()
    assert out[0][0] == out[1][0]
    for x, y in zip(out[0][1:], out[1][1:]):
        assert np.abs(x - y).max() <= 1e-8 * np.abs(x).max()


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


@pytest.mark.gpu
@pytest.mark.parametrize("place", [0, 0.4, 1.0])
def test_bad_entries_are_refused_before_the_device(place):
    """The same on the device path: refused by the upload, on the host, and
    the next upload of the subdomain is taken."""
    print("case bad entries", place, flush=True)
    p = CubeProblem(8, 2, rhs="random", seed=3)
    subs = list(p.subdomains())
    d = subs[0]
    k = int(place * (len(d["a_sparse"]) - 1))
    b = bddcml_amd.Bddcml()
    b.init(2, [p.nsub, 1], numbase=p.numbase)
    for i, j, text in ((5, 3, "upper triangle"), (1, d["ndofs"] + 1, "out of range"),
                       (0, 3, "out of range")):
        bad = dict(d, i_sparse=d["i_sparse"].copy(), j_sparse=d["j_sparse"].copy())
        bad["i_sparse"][k], bad["j_sparse"][k] = i, j
        with pytest.raises(RuntimeError, match=text):
            b.upload_subdomain_data(bad)
    for s in subs:
        b.upload_subdomain_data(s)
    b.setup_preconditioner()
    assert b.solve(0, 1e-8, 100, 50)[1] == 0
    b.finalize()


@pytest.mark.gpu
@pytest.mark.parametrize("nel", [4, 8])
def test_plan_only_after_the_uploads(nel):
    """plan_only set between the uploads and the setup: the plan has the
    diagonals (stiffness weights) and patterns that were assembled on the
    device, as a plan from host assemblies and a whole setup have."""
    print("case plan after uploads", nel, flush=True)
    p = CubeProblem(nel, 2, rhs="random", seed=3, dirichlet="random")
    out = []
    for before, after in ((0, 1), (1, 1), (0, 0)):
        b = bddcml_amd.Bddcml()
        b.init(2, [p.nsub, 1], numbase=p.numbase)
        b.set_option("plan_only", before)
        for d in p.subdomains():
            b.upload_subdomain_data(d)
        b.set_option("plan_only", after)
        b.setup_preconditioner(1, weights_type=1)
        maps = [b.sub_maps(s + p.numbase) for s in range(p.nsub)]
        out.append((b.counts(), [x for m in maps for x in m], b.interface_dofs()))
        b.finalize()
    for c, maps, dofs in out[1:]:
        assert c == out[0][0] and np.array_equal(dofs, out[0][2])
        assert all(np.array_equal(x, y) for x, y in zip(maps, out[0][1]))


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
