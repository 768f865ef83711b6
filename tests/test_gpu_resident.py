"""The resident form of a single dense instance (xcs_resident.h) where it can go
wrong: row tiles of one float4 and of the largest kind, workgroups without rows,
odd row and column counts, the largest n that fits its LDS and the first that
does not (general form), a whole-support (Gaussian) run and k = 0, each against
the general one-workgroup form on the same generated instance and the planted
signal."""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu

TOL = 1e-5


def _solve(ga, alg, k, m, n, **kw):
    pl = ga.Plan(alg, "gen", k, m, n, 0, ga.options(tol=TOL, seed=20260101, **kw))
    pl.solve()
    r = pl.results()
    r["geometry"] = pl.geometry()
    pl.solve()
    again = pl.results()["x"]
    pl.close()
    np.testing.assert_array_equal(r["x"], again)  # fixed order of every sum
    return r


@pytest.mark.parametrize("alg", ["NIHT", "HTP", "CGIHT"])
@pytest.mark.parametrize("k,m,n,team,block", [
    (20, 256, 1024, 64, 512),    # one float4 of rows per workgroup
    (20, 256, 1024, 128, 256),   # half the workgroups without rows
    (9, 255, 777, 2, 512),       # odd sizes, tiles of 128 rows
    (9, 193, 1025, 16, 1024),    # n one past a whole word of the mask
    (40, 1001, 2501, 48, 512),   # a team that is no multiple of 16
    (60, 1000, 9000, 0, 0),      # close to the LDS limit
    (60, 1000, 11000, 0, 0),     # beyond it: the general form
    (30, 3000, 700, 16, 512),    # m > n
])
def test_resident_matches_general_form(lib, alg, k, m, n, team, block):
    kw = {}
    if team:
        kw["teamSize"] = team
    if block:
        kw["blockSize"] = block
    a = _solve(lib, alg, k, m, n, **kw)
    b = _solve(lib, alg, k, m, n, teamSize=1, blockSize=512)
    if team:
        assert a["geometry"] == (team, block)
    # both stop at |r| <= tol: |x - x_true| <= tol / sigma with the smallest singular
    # value on 2k columns above 1 / 3 at these densities, and |x_true| = sqrt(k)
    bound = 3 * TOL / np.sqrt(k)
    for r in (a, b):
        assert np.linalg.norm(r["x"] - r["x_true"]) <= bound * np.linalg.norm(r["x_true"])
    assert a["stop_reason"] == b["stop_reason"] == 0
    assert abs(a["iters"] - b["iters"]) <= 1


def test_resident_dense_support_and_plain_form(lib):
    """Gaussian values: the bins keep most entries at times.  The host-stepped form
    saves and reloads the state every iteration: the same bits."""
    for alg in ("NIHT", "HTP", "CGIHT"):
        a = _solve(lib, alg, 30, 600, 2400, vecDistribution="gaussian", instance=3)
        b = _solve(lib, alg, 30, 600, 2400, vecDistribution="gaussian", instance=3, mode=1)
        np.testing.assert_array_equal(a["x"], b["x"])
        assert a["iters"] == b["iters"] and a["stop_reason"] == b["stop_reason"]
        assert np.abs(a["x"] - a["x_true"]).max() < 1e-3 * np.abs(a["x_true"]).max()


def test_resident_empty_support(lib):
    a = _solve(lib, "CGIHT", 0, 256, 1024, maxiter=20, teamSize=16)
    assert not a["x"].any()
