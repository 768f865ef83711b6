"""The split form of a single sparse or DCT instance (xcs_split.h) where it can
go wrong: odd sizes, slices shorter than the rest, workgroups without rows, even
and odd powers of two (equal and unequal transform factors), the smallest and
largest teams of a transform, histograms beyond the LDS one, sizes it refuses
(general form) and k = 0, against the general one-workgroup form on the same
generated instance and the planted signal."""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu

TOL = 1e-5


def _solve(ga, alg, ens, k, m, n, p, **kw):
    if ens == "smv":
        kw["matrixEnsemble"] = "binary"
    pl = ga.Plan(alg, ens, k, m, n, p, ga.options(tol=TOL, seed=20260101, **kw))
    pl.solve()
    r = pl.results()
    r["geometry"] = pl.geometry()
    pl.solve()
    np.testing.assert_array_equal(r["x"], pl.results()["x"])  # fixed order of every sum
    pl.close()
    return r


@pytest.mark.parametrize("alg", ["NIHT", "HTP", "CGIHT"])
@pytest.mark.parametrize("ens,k,m,n,p,team,extra", [
    ("smv", 9, 333, 1001, 7, 2, {}),
    ("smv", 9, 333, 1001, 7, 30, {}),      # trailing workgroups without columns
    ("smv", 40, 1000, 4001, 3, 16, {"blockSize": 256}),
    ("smv", 40, 600, 4001, 20, 64, {}),    # long rows: eight lanes each
    ("smv", 60, 2000, 8191, 7, 0, {"numBins": 5000}),  # bins in memory, the extra hop
    ("dct", 9, 200, 512, 0, 2, {}),        # 16 x 16
    ("dct", 9, 200, 512, 0, 8, {}),        # its largest team
    ("dct", 12, 401, 1024, 0, 4, {}),      # 16 x 32
    ("dct", 30, 1501, 8192, 0, 0, {"numBins": 5000}),
    ("dct", 9, 200, 512, 0, 16, {}),       # more than the factors allow: general form
    ("dct", 9, 200, 512, 0, 3, {}),        # no power of two: general form
])
def test_split_matches_general_form(lib, alg, ens, k, m, n, p, team, extra):
    kw = dict(extra)
    if team:
        kw["teamSize"] = team
    a = _solve(lib, alg, ens, k, m, n, p, **kw)
    kw.update(teamSize=1, blockSize=512)
    b = _solve(lib, alg, ens, k, m, n, p, **kw)
    if team:
        assert a["geometry"][0] == team
    # both stop at |r| <= tol: |x - x_true| <= tol / sigma with the smallest singular
    # value on 2k columns above 1 / 3 at these densities, and |x_true| = sqrt(k)
    bound = 3 * TOL / np.sqrt(k)
    for r in (a, b):
        assert np.linalg.norm(r["x"] - r["x_true"]) <= bound * np.linalg.norm(r["x_true"])
    assert a["stop_reason"] == b["stop_reason"] == 0
    assert abs(a["iters"] - b["iters"]) <= 1


@pytest.mark.parametrize("ens,m,n,p", [("smv", 700, 2400, 7), ("dct", 700, 2048, 0)])
@pytest.mark.parametrize("alg", ["NIHT", "HTP", "CGIHT"])
@pytest.mark.parametrize("restart", [0, 1])
def test_split_plain_form_and_dense_support(lib, ens, m, n, p, alg, restart):
    """Gaussian values: the bins keep most entries at times.  The host-stepped form
    saves and reloads the state every iteration: the same bits."""
    kw = dict(vecDistribution="gaussian", instance=3, restartFlag=restart)
    a = _solve(lib, alg, ens, 30, m, n, p, **kw)
    b = _solve(lib, alg, ens, 30, m, n, p, mode=1, **kw)
    np.testing.assert_array_equal(a["x"], b["x"])
    assert a["iters"] == b["iters"] and a["stop_reason"] == b["stop_reason"]
    assert np.abs(a["x"] - a["x_true"]).max() < 1e-3 * np.abs(a["x_true"]).max()


@pytest.mark.parametrize("ens,p", [("smv", 7), ("dct", 0)])
def test_split_empty_support(lib, ens, p):
    assert not _solve(lib, "CGIHT", ens, 0, 256, 1024, p, maxiter=20)["x"].any()
