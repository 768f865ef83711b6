"""The many-RHS solver's per-signal kernels and product shapes at their edges: one
signal, the smallest m, rows beyond the small residual kernel, n beyond what the
selection holds in LDS, a histogram beyond the LDS one, restarts, and ties at the
k-th magnitude, against the planted signals.  The refinement leaves least squares
on the support (its FP64 residual below tol), so |x - x_true| <= tol / sigma with
the smallest singular value on 2k columns above 1 / 3."""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu

TOL = 1e-5


@pytest.mark.parametrize("precision", ["bf16", "fp8"])
@pytest.mark.parametrize("m,n,k,count,extra", [
    (128, 512, 6, 1, {}),
    (128, 512, 6, 130, {}),
    (256, 1024, 12, 33, {"numBins": 5000}),
    (256, 1024, 12, 33, {"restartFlag": 1}),
    (640, 16896, 12, 5, {}),            # n past the LDS selection
    (4224, 8704, 80, 3, {}),            # m past the 4-float4 residual kernel
    (512, 2048, 20, 257, {"vecDistribution": "binary"}),  # magnitudes near ties
])
def test_recovers(lib, precision, m, n, k, count, extra):
    opts = dict(tol=TOL, seed=20260101, vecDistribution="gaussian")
    opts.update(extra)
    R = lib.ManyRHS(m, n, k, count, precision, lib.options(**opts))
    R.solve()
    r = R.results()
    first = [R.x(s)[0].copy() for s in range(min(count, 8))]
    good = r["norms"][:, 2] < 1e-3
    assert good.mean() >= 0.97, good.mean()
    for s in range(min(count, 40)):
        x, xt, y = R.x(s)
        assert (x != 0).sum() <= k
        if good[s]:
            assert np.linalg.norm(x - xt) <= 3 * TOL
            assert r["resid_rel"][s] * np.linalg.norm(y.astype(np.float64)) <= TOL
    R.solve()
    for s, x in enumerate(first):
        np.testing.assert_array_equal(R.x(s)[0], x)  # fixed order of every sum
    R.close()
