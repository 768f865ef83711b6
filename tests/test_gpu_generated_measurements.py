"""A generated instance's measurements come from the product its solves use: the
planted vector then leaves no residual at all, so a solve gets below the rounding
of the measurements themselves, ||y|| 2^-24, and a tolerance near that is met
instead of ending in a stall."""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("alg", ["NIHT", "HTP"])
@pytest.mark.parametrize("ens,k,m,n,p,extra", [
    ("gen", 20, 256, 1024, 0, {}),
    ("gen", 50, 1024, 4096, 0, {}),
    ("gen", 50, 1024, 4096, 0, {"blockSize": 1024}),
    ("gen", 30, 700, 2001, 0, {"teamSize": 48}),
    ("smv", 300, 4000, 20000, 7, {}),
    ("dct", 100, 2049, 8192, 0, {}),
    ("dct", 1000, 32769, 131072, 0, {}),
])
def test_solves_below_the_rounding_of_y(lib, alg, ens, k, m, n, p, extra):
    kw = dict(extra, seed=77, maxiter=60)
    if ens == "smv":
        kw["matrixEnsemble"] = "binary"
    first = lib.Plan(alg, ens, k, m, n, p, lib.options(tol=1.0, **kw))
    first.solve()
    y = float(first.trace(1)[1][0])  # the residual of x = 0
    first.close()
    pl = lib.Plan(alg, ens, k, m, n, p, lib.options(tol=y * 2.0 ** -24, **kw))
    pl.solve()
    r = pl.results()
    pl.close()
    assert r["stop_reason"] == 0
    # |x - x_true| <= tol / sigma, the smallest singular value on 2k columns above 1 / 4
    # (a quarter of an orthogonal matrix's rows has scale 1 / 2), |x_true| = sqrt(k)
    err = np.linalg.norm(r["x"].astype(np.float64) - r["x_true"])
    assert err <= 4 * y * 2.0 ** -24


@pytest.mark.parametrize("alg", ["NIHT", "HTP", "CGIHT"])
def test_large_transform_meets_its_tolerance(lib, alg):
    """1.7e-7 of ||y||: the general form's measurements left 1.15e-5 here."""
    pl = lib.Plan(alg, "dct", 13107, (1 << 18) + 1, 1 << 20, 0, lib.options(tol=1e-5, seed=77, maxiter=60))
    pl.solve()
    r = pl.results()
    pl.close()
    assert r["stop_reason"] == 0
