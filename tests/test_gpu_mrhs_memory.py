"""The many-RHS exact residual where its row-blocked copy of A is longer than 32-bit
offsets reach, and where there is no memory for that copy at all."""
import ctypes

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


def test_without_memory_for_the_row_blocked_copy(lib):
    hip = ctypes.CDLL("libamdhip64.so")
    free, total = ctypes.c_size_t(), ctypes.c_size_t()

    def left():
        assert hip.hipMemGetInfo(ctypes.byref(free), ctypes.byref(total)) == 0
        return free.value
    m, n, k, count = 4096, 16384, 100, 4
    copy = 4 * m * n

    def make():
        R = lib.ManyRHS(m, n, k, count, "bf16", lib.options(tol=1e-5, seed=3, vecDistribution="gaussian"))
        R.solve()
        return R, np.stack([R.x(s)[0] for s in range(count)]), R.results()
    before = left()
    R, x, r = make()
    used = before - left()
    R.close()
    assert used > 3 * copy  # A in FP32 twice, two BF16 copies of half the size
    ballast = []
    try:
        while left() > used - copy // 2:  # room for everything but the copy
            p = ctypes.c_void_p()
            want = min(left() - (used - copy // 2), 16 << 30)
            if want < 1 << 21:
                break
            if hip.hipMalloc(ctypes.byref(p), ctypes.c_size_t(want)) != 0:
                break
            ballast.append(p)
        assert left() < used - copy // 4
        R, x2, r2 = make()
        assert left() < copy  # the handle lies beside the ballast, without room for the copy
        R.close()
    finally:
        for p in ballast:
            hip.hipFree(p)
    np.testing.assert_array_equal(x2, x)  # the same sums in the same order
    np.testing.assert_array_equal(r2["resid_rel"], r["resid_rel"])
    assert (r["norms"][:, 2] < 1e-3).all()
