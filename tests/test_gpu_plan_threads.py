"""One plan read by several threads at once: every reader gets the solution, the
planted vector and the errors of the last solve, with the solution in the plan's
staging memory and past it."""
import threading

import numpy as np
import pytest

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("n", [4096, 1 << 16, 1 << 17])
def test_concurrent_readers(lib, n):
    pl = lib.Plan("NIHT", "dct", n // 200, n // 4, n, 0, lib.options(tol=1e-5, seed=4, maxiter=8))
    pl.solve()
    want = pl.results()
    bad = []

    def work():
        for _ in range(40):
            r = pl.results()
            if not (np.array_equal(r["x"], want["x"]) and np.array_equal(r["x_true"], want["x_true"]) and
                    np.array_equal(r["norms"], want["norms"]) and np.array_equal(r["support"], want["support"])):
                bad.append(1)
    th = [threading.Thread(target=work) for _ in range(8)]
    [t.start() for t in th]
    [t.join() for t in th]
    pl.close()
    assert not bad


def test_readers_beside_a_solve(lib):
    """Solves of one plan give the same bits every time, so a reader beside them sees
    either the planted instance's start, a state between, or the solution; what it
    gets after the last solve is that solve's."""
    pl = lib.Plan("NIHT", "gen", 20, 256, 1024, 0, lib.options(tol=1e-5, seed=4))
    pl.solve()
    want = pl.results()["x"]
    stop = threading.Event()

    def work():
        while not stop.is_set():
            pl.results()
    th = [threading.Thread(target=work) for _ in range(4)]
    [t.start() for t in th]
    for _ in range(50):
        pl.solve()
    stop.set()
    [t.join() for t in th]
    assert np.array_equal(pl.results()["x"], want)
    pl.close()
