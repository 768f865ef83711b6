"""Which form a plan's solves run in, and each branch of the forms with the sizes
that really reach it, against the general one-workgroup form on the same generated
instance and the planted signal."""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu

TOL = 1e-5


def _solve(ga, alg, ens, k, m, n, p=0, **kw):
    if ens == "smv":
        kw["matrixEnsemble"] = "binary"
    pl = ga.Plan(alg, ens, k, m, n, p, ga.options(tol=TOL, seed=20260101, maxiter=200, **kw))
    pl.solve()
    r = pl.results()
    r["form"], r["geometry"] = pl.form(), pl.geometry()
    pl.close()
    return r


def _agree(a, b, k):
    # both stop at |r| <= tol: |x - x_true| <= tol / sigma with the smallest singular
    # value on 2k columns above 1 / 3 at these densities, and |x_true| = sqrt(k)
    bound = 3 * TOL / np.sqrt(k)
    for r in (a, b):
        assert np.linalg.norm(r["x"] - r["x_true"]) <= bound * np.linalg.norm(r["x_true"])
    assert a["stop_reason"] == b["stop_reason"] == 0
    assert abs(a["iters"] - b["iters"]) <= 1


def _resident_bytes(n, lda, bins):
    """LDS of the resident form: x, g, p, r, histogram, two masks, a 16-bit list."""
    up = lambda b: (b + 15) // 16 * 16  # noqa: E731
    return 3 * up(4 * n) + up(4 * lda) + up(4 * bins) + 2 * up(8 * (n // 64 + 1)) + up(2 * n)


@pytest.mark.parametrize("alg", ["NIHT", "HTP", "CGIHT"])
def test_resident_at_its_largest_n_and_past_it(lib, alg):
    m, lda, k = 1000, 1024, 60
    n = max(q for q in range(9000, 11000) if _resident_bytes(q, lda, max(q // 20, 1000)) <= 144 * 1024)
    for size, form in ((n, "resident"), (n + 8, "general")):
        a = _solve(lib, alg, "gen", k, m, size)
        assert a["form"] == (form, False, 0, 0)
        _agree(a, _solve(lib, alg, "gen", k, m, size, teamSize=1, blockSize=512), k)


@pytest.mark.parametrize("alg", ["NIHT", "HTP", "CGIHT"])
@pytest.mark.parametrize("k,m,n,team", [(20, 256, 1024, 64), (60, 1000, 9000, 0), (30, 3000, 700, 16),
                                         (40, 1001, 2501, 48)])
def test_resident_with_1024_threads(lib, alg, k, m, n, team):
    kw = dict(teamSize=team) if team else {}
    a = _solve(lib, alg, "gen", k, m, n, blockSize=1024, **kw)
    assert a["form"][0] == "resident" and a["geometry"][1] == 1024
    _agree(a, _solve(lib, alg, "gen", k, m, n, teamSize=1, blockSize=512), k)


@pytest.mark.parametrize("k,m,n,kw", [(30, 600, 2400, {}), (60, 1000, 9000, {}), (30, 600, 2400, {"blockSize": 1024})])
def test_resident_with_restarts(lib, k, m, n, kw):
    """restartFlag: a lost support entry starts the directions anew; the host-stepped
    form saves and reloads that state every iteration: the same bits."""
    a = _solve(lib, "CGIHT", "gen", k, m, n, restartFlag=1, **kw)
    assert a["form"][0] == "resident"
    _agree(a, _solve(lib, "CGIHT", "gen", k, m, n, restartFlag=1, teamSize=1, blockSize=512), k)
    b = _solve(lib, "CGIHT", "gen", k, m, n, restartFlag=1, mode=1, **kw)
    np.testing.assert_array_equal(a["x"], b["x"])
    assert a["iters"] == b["iters"]


@pytest.mark.parametrize("algs,k,m,n,p,team,bits,rows,cols", [
    (("NIHT", "HTP", "CGIHT"), 20, 400, 65536, 7, 128, True, 128, 128),  # rows of 1147 entries
    (("NIHT", "CGIHT"), 40, 1500, 40000, 9, 4, True, 0, 0),         # support bits in LDS, the entries in memory
    (("HTP",), 40, 1500, 30000, 9, 4, True, 0, 0),                  # the same beside a fourth slice
    (("NIHT", "CGIHT"), 60, 20000, 1 << 19, 7, 256, True, 256, 0),  # the rows' entries in LDS, the columns' in memory
    (("HTP",), 60, 20000, 1 << 19, 6, 256, True, 256, 0),
    (("NIHT", "HTP", "CGIHT"), 60, 20000, 1 << 20, 6, 256, False, 0, 0),  # no room for the support bits
    (("NIHT", "HTP", "CGIHT"), 60, 1100, 16384, 7, 16, True, 16, 16),     # two columns and more a thread
])
def test_split_stages_what_fits(lib, algs, k, m, n, p, team, bits, rows, cols):
    for alg in algs:
        a = _solve(lib, alg, "smv", k, m, n, p, teamSize=team, blockSize=512)
        assert a["form"][:2] == ("split", bits), alg
        # a few workgroups may differ from the rest: rows are drawn, not dealt
        assert abs(a["form"][2] - rows) <= team // 16 and abs(a["form"][3] - cols) <= team // 16, a["form"]
        _agree(a, _solve(lib, alg, "smv", k, m, n, p, teamSize=1, blockSize=512), k)


@pytest.mark.parametrize("alg,ens,k,m,n,p,kw,form", [
    ("HTP", "smv", 40, 1500, 40000, 9, {"teamSize": 4}, "general"),  # four slices of 10 048 do not fit
    ("FIHT", "gen", 20, 256, 1024, 0, {}, "general"),
    ("NIHT", "gen", 20, 256, 1024, 0, {"timing": "on"}, "general"),
    ("NIHT", "gen", 20, 256, 1024, 0, {"teamSize": 1}, "general"),
    ("NIHT", "gen", 20, 256, 1024, 0, {"teamSize": 2}, "resident"),
    ("NIHT", "smv", 9, 333, 1001, 7, {"teamSize": 1}, "general"),
    ("NIHT", "smv", 9, 333, 900, 7, {}, "general"),        # 1000 bins for 900 entries
    ("NIHT", "smv", 9, 333, 1001, 7, {}, "split"),
    ("NIHT", "smv", 60, 2000, 8191, 7, {"blockSize": 1024}, "general"),
    ("NIHT", "dct", 9, 200, 1024, 0, {"teamSize": 3}, "general"),
    ("NIHT", "dct", 9, 200, 1024, 0, {"teamSize": 8}, "split"),
    ("NIHT", "dct", 9, 200, 1024, 0, {"teamSize": 16}, "general"),  # more than half the 16 rows
])
def test_the_form_of_a_plan(lib, alg, ens, k, m, n, p, kw, form):
    a = _solve(lib, alg, ens, k, m, n, p, **kw)
    assert a["form"][0] == form
    assert a["stop_reason"] == 0 and a["norms"][2] < 1e-3
