"""The schedule of the IC(0) sweeps (host only): every value read after it is
written and before its place in the LDS ring is reused, over chains, bands,
plates, blocks and random patterns, and a stream of at most a small multiple of
the factor's bytes."""
import numpy as np
import pytest
import scipy.sparse as sp

from rustyfem_amd import ffi, meshes


def lower_csc(a):
    low = sp.csc_matrix(sp.tril(sp.csc_matrix(a)))
    low.sort_indices()
    return low.indptr.astype(np.int64), low.indices.astype(np.int64)


def chain(n):
    return sp.diags([-1.0, 2.5, -1.0], [-1, 0, 1], shape=(n, n), format="csc")


def band(n, w):
    return sp.diags([np.ones(n - k) for k in range(w + 1)], list(range(0, -w - 1, -1)), shape=(n, n), format="csc")


def random_lower(n, per_row, reach, seed, dofs=1):
    """About per_row entries a row, up to `reach` rows back, in blocks of `dofs` rows."""
    rng = np.random.default_rng(seed)
    r = np.repeat(np.arange(n), per_row)
    c = np.maximum(0, r - rng.integers(0, reach + 1, n * per_row))
    a = sp.csc_matrix((np.ones(len(r)), (r, c)), shape=(n, n)) + sp.identity(n)
    return sp.kron(a, np.ones((dofs, dofs)), format="csc")


CASES = {"hex3": lambda: meshes.hex_block(3).to_scipy(), "hex18": lambda: meshes.hex_block(18).to_scipy(),
         "hex60x2x3": lambda: meshes.hex_block(60, 2, 3).to_scipy(),
         "tet9": lambda: meshes.tet_block(9, seed=2).to_scipy(),
         "plate31x9": lambda: meshes.plate_cpe4(31, 9, 1e11, 0.3, nrhs=1).to_scipy(),
         "plate120x90": lambda: meshes.plate_cpe4(120, 90, 1e11, 0.3, nrhs=1).to_scipy(),
         "laplace16": lambda: meshes.laplacian3d(16).to_scipy(), "chain400": lambda: chain(400),
         "chain4001": lambda: chain(4001), "band2000_7": lambda: band(2000, 7), "band700_60": lambda: band(700, 60),
         "one": lambda: chain(1), "diagonal": lambda: sp.identity(129, format="csc"),
         "random1": lambda: random_lower(3000, 4, 40, 1), "random2": lambda: random_lower(1100, 3, 25, 2, 2),
         "random3": lambda: random_lower(900, 6, 60, 3, 3), "random_wide": lambda: random_lower(6000, 2, 1500, 4),
         "random4": lambda: random_lower(400, 5, 30, 5, 4)}


@pytest.mark.parametrize("case", sorted(CASES))
def test_schedule_is_sound(case):
    low = lower_csc(CASES[case]())
    n = len(low[0]) - 1
    dirs, what = ffi.sweep_plan(n, *low)
    assert what == ""
    for d in dirs:
        if d["rows"]:
            assert d["reach"] < d["ring"] and d["row_levels"] >= d["levels"] >= 1 and d["rounds"] >= d["levels"]
    if all(d["rows"] for d in dirs) and n > 1:
        assert ffi.sweep_plan(n, *low, plant=2)[1] != ""
        if dirs[0]["levels"] > 1:
            assert ffi.sweep_plan(n, *low, plant=1)[1] != ""


def test_sweeps_are_taken_where_they_were_measured():
    for make, rows in ((lambda: meshes.hex_block(12).to_scipy(), 3), (lambda: chain(1000), 1),
                       (lambda: meshes.plate_cpe4(60, 6, 1e11, 0.3, nrhs=1).to_scipy(), 2)):
        low = lower_csc(make())
        dirs, what = ffi.sweep_plan(len(low[0]) - 1, *low)
        assert what == "" and [d["rows"] for d in dirs] == [rows, rows]


@pytest.mark.parametrize("case", ["chain", "beam", "band"])
def test_stream_is_bounded_by_the_factor(case):
    """One group per level fills one of the 64 slots of a round: a chain of
    10^6 rows (12 MB of factor) would stream 16 GB.  The stream stays below 256 MB
    and 16 times the factor (12 bytes an entry, 16 a row), else there is no sweep."""
    a = {"chain": lambda: chain(1_000_000), "beam": lambda: meshes.hex_block(3000, 1, 1).to_scipy(),
         "band": lambda: band(200_000, 2)}[case]()
    low = lower_csc(a)
    n, nnz = len(low[0]) - 1, len(low[1]) - (len(low[0]) - 1)
    dirs, what = ffi.sweep_plan(n, *low)
    assert what == ""
    for d in dirs:
        assert d["bytes"] <= 256e6 + 16 * (12 * nnz + 16 * n)
    if case != "beam":
        assert [d["rows"] for d in dirs] == [0, 0]


def test_unsorted_pattern_is_refused():
    with pytest.raises(RuntimeError):
        ffi.sweep_plan(2, np.array([0, 2, 3]), np.array([1, 0, 1]))
