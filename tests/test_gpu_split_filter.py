"""Sparse products of the split form that read the support only (xcs_split.h):
with the entries staged in LDS in full, in part or not at all, without room for
the support bits, with rows longer than one block of tested entries, and with
empty and uneven rows and columns, against the general one-workgroup form."""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu

TOL = 1e-5


def _close(a, b, k):
    # both stop at |r| <= tol: |x - x_true| <= tol / sigma with the smallest singular
    # value on 2k columns above 1 / 3 at these densities, and |x_true| = sqrt(k)
    bound = 3 * TOL / np.sqrt(k)
    return np.linalg.norm(a - b) <= bound * np.linalg.norm(b)


@pytest.mark.parametrize("alg", ["NIHT", "HTP", "CGIHT"])
@pytest.mark.parametrize("k,m,n,p,team", [
    (20, 400, 65536, 7, 128),       # 1147 entries a row: more than 64 for each of 16 lanes
    (40, 1500, 40000, 9, 4),        # support bits in LDS, the entries in memory
    (60, 20000, 1 << 19, 7, 256),   # the rows' entries in LDS, the columns' in memory
    (60, 20000, 1 << 20, 6, 256),   # no room for the support bits
    (30, 2000, 8191, 1, 8),         # one entry a column
    (60, 1100, 16384, 7, 16),       # two columns and more a thread
])
def test_products_on_the_support(lib, alg, k, m, n, p, team):
    out = []
    for t in (team, 1):
        pl = lib.Plan(alg, "smv", k, m, n, p,
                      lib.options(tol=TOL, seed=20260101, matrixEnsemble="binary", teamSize=t, blockSize=512,
                                  maxiter=200))
        pl.solve()
        r = pl.results()
        pl.solve()
        np.testing.assert_array_equal(r["x"], pl.results()["x"])
        pl.close()
        out.append(r)
    a, b = out
    if p > 1:  # a single entry a column: rows collide, the planted vector need not be found
        assert _close(a["x"], a["x_true"], k) and _close(b["x"], b["x_true"], k)
        assert a["stop_reason"] == b["stop_reason"] == 0
    assert abs(a["iters"] - b["iters"]) <= 1


@pytest.mark.parametrize("alg", ["NIHT", "HTP", "CGIHT"])
def test_uneven_rows_and_columns(lib, alg):
    rng = np.random.default_rng(8)
    m, n, k = 700, 3000, 12
    rows, cols, vals = [], [], []
    for j in range(n):
        c = 0 if j % 97 == 5 else int(rng.integers(1, 40))  # some columns empty
        r = rng.choice(m - 60, c, replace=False)            # the last 60 rows empty
        rows += list(r)
        cols += [j] * c
        vals += list(rng.choice([-1.0, 1.0], c) / np.sqrt(max(c, 1)))
    # a last column with an entry, so that n is what the call finds
    rows, cols, vals = np.array(rows + [0]), np.array(cols + [n - 1]), np.array(vals + [0.0], np.float32)
    x = np.zeros(n)
    live = [j for j in rng.permutation(n) if j % 97 != 5][:k]
    x[live] = 1.0
    y = np.zeros(m)
    np.add.at(y, rows, vals.astype(np.float64) * x[cols])
    got = [lib.cs(alg, "smv", y.astype(np.float32), rows + 1, cols + 1, vals, k,
                  lib.options(tol=TOL, teamSize=t, blockSize=512))[0] for t in (16, 64, 1)]
    for g in got:
        assert _close(g, x, k)
