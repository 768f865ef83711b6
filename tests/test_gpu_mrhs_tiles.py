"""Products of the many-RHS solver: the block tile, chosen or left to the sizes again,
does not change a bit of a solution; the same signals beside fewer or more others
end within their tolerance of each other."""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu

TOL = 1e-5


def _solve(R, count):
    R.solve()
    return np.stack([R.x(s)[0] for s in range(count)])


@pytest.mark.parametrize("precision", ["bf16", "fp8"])
@pytest.mark.parametrize("m,n,k,count", [(512, 2048, 20, 200), (1024, 4096, 50, 40), (384, 1024, 12, 130)])
def test_tiles_give_the_same_bits(lib, precision, m, n, k, count):
    R = lib.ManyRHS(m, n, k, count, precision, lib.options(tol=TOL, seed=20260101, vecDistribution="gaussian"))
    want = _solve(R, count)
    assert (R.results()["norms"][:, 2] < 1e-3).mean() > 0.95
    for tile in (0, 1, 2, -1):
        R.gemm_tile(tile)
        np.testing.assert_array_equal(_solve(R, count), want)
    for tile in (-2, 3):
        with pytest.raises(lib.GagaError, match="tile must be"):
            R.gemm_tile(tile)
    R.close()


@pytest.mark.parametrize("precision", ["bf16", "fp8"])
def test_the_same_signals_among_others(lib, precision):
    out = []
    for count in (8, 60, 300):
        R = lib.ManyRHS(512, 2048, 20, count, precision,
                        lib.options(tol=TOL, seed=20260101, vecDistribution="gaussian"))
        x = _solve(R, 8)
        out.append((x, R.results()["norms"][:8, 2] < 1e-3))
        R.close()
    for x, good in out[1:]:
        for s in range(8):
            # both at |r| <= tol: |x - x_true| <= tol / sigma each, the smallest singular value on
            # 2k columns above 1 / 3
            if good[s] and out[0][1][s]:
                assert np.linalg.norm(x[s] - out[0][0][s]) <= 6 * TOL
    assert all(g.sum() >= 7 for _, g in out)
