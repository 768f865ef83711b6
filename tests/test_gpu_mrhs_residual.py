"""The many-RHS solver's exact residual where its row blocks and lists have edges:
fewer row blocks than XCDs, the most rows, supports beyond one LDS list, one
signal and many, all signals and the active ones, against 64-bit sums on the host
over the same matrix and the returned vectors."""
import numpy as np
import pytest

from gaga_amd import _capi

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("m,n,k,count,corrections", [
    (128, 512, 6, 1, 2),          # four row blocks for eight XCDs
    (384, 1024, 17, 40, 6),       # twelve
    (8192, 8704, 30, 2, 2),       # the most rows
    (2048, 4096, 1100, 3, 1),     # a support list in two parts
    (1024, 2048, 1024, 2, 0),     # exactly one whole list
    (256, 1024, 13, 600, 6),      # several groups' worth of signals
])
def test_exact_residual(lib, m, n, k, count, corrections):
    seed = 20260101
    R = lib.ManyRHS(m, n, k, count, "bf16",
                    lib.options(tol=1e-6, seed=seed, maxiter=12, vecDistribution="gaussian"))
    R.configure(corrections=corrections)
    R.solve()
    rel = R.results()["resid_rel"]
    A = _capi.generate_gen(m, n, seed, 0).astype(np.float64)  # row j = column j
    for s in sorted({0, count // 2, count - 1}):
        x, _, y = R.x(s)
        y = y.astype(np.float64)
        ref = np.linalg.norm(y - x.astype(np.float64) @ A) / np.linalg.norm(y)
        # sums of k products, each rounded once, against sums in another order
        assert abs(rel[s] - ref) <= 4 * (k + 2) * 2.0 ** -53 * np.sqrt(m) + 1e-12 * ref, (s, rel[s], ref)
    R.close()
