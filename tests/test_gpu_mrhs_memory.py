"""The many-RHS exact residual where its row-blocked copy of A is longer than 32-bit
offsets reach, and without that copy (a handle does without where there is no memory
for it)."""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu


def test_columns_beyond_32_bit_offsets(lib):
    # 128-byte pieces: offsets beyond 2^32 from column 2^25 on; half of the signals have theirs there
    n, count = 1 << 26, 8
    R = lib.ManyRHS(128, n, 1, count, "bf16",
                    lib.options(tol=1e-5, seed=3, vecDistribution="gaussian", maxiter=50))
    R.solve()
    r = R.results()
    true = [R.x(s)[1] for s in range(count)]
    assert any(np.flatnonzero(t)[0] >= 1 << 25 for t in true)
    for s in range(count):
        x = R.x(s)[0]
        assert np.array_equal(np.flatnonzero(x), np.flatnonzero(true[s]))
        # one column of unit length: |x - x_true| <= |r| / |a| with |a| > 1 / 2
        assert np.abs(x - true[s]).max() <= 2e-5 and r["resid_rel"][s] <= 1e-6
    R.close()


@pytest.mark.parametrize("m,n,k,count", [(128, 512, 6, 3), (4096, 16384, 100, 4), (1024, 4096, 50, 300)])
def test_without_the_row_blocked_copy(lib, m, n, k, count):
    R = lib.ManyRHS(m, n, k, count, "bf16", lib.options(tol=1e-5, seed=3, vecDistribution="gaussian"))
    out = []
    for keep in (True, False, False, True):
        R.row_blocks(keep)
        R.solve()
        out.append((np.stack([R.x(s)[0] for s in range(count)]), R.results()))
    R.close()
    for x, r in out[1:]:
        np.testing.assert_array_equal(x, out[0][0])  # the same sums in the same order
        np.testing.assert_array_equal(r["resid_rel"], out[0][1]["resid_rel"])
    assert (out[0][1]["norms"][:, 2] < 1e-3).mean() > 0.95
