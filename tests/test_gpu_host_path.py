"""The host side of a call: solution vectors read in any order hold the same
bits, the relative errors that the device sums match 64-bit sums on the host,
and calls from several threads do not disturb each other."""
import threading

import numpy as np
import pytest

import gaga_amd as ga

pytestmark = pytest.mark.gpu


def _order(count):
    """Every index at least once: in order from the middle, backwards, strided, in order."""
    idx = list(range(count // 2, count)) + list(range(count - 1, -1, -3)) + [0, 1, 0, 1, 2, 3]
    return [i for i in idx if i < count] + list(range(count))


def _check_reads(h, count, pieces):
    # a descending read is never in order: each vector comes by its own copy
    alone = {i: [a.copy() for a in pieces(h.x(i))] for i in range(count - 1, -1, -1)}
    for i in _order(count):
        for a, b in zip(pieces(h.x(i)), alone[i]):
            assert np.array_equal(a, b), i
    return alone


@pytest.mark.parametrize("count", [1, 2, 150])
def test_batch_reads(count):
    specs = [dict(ens="gen" if i % 3 else "smv", k=3 + i % 5, m=40 + i % 7, n=101 + 13 * (i % 11), p=7, instance=i)
             for i in range(count)]
    B = ga.Batch("NIHT", specs, ga.options(tol=1e-6, seed=3))
    B.solve()
    alone = _check_reads(B, count, lambda r: r)
    assert any(np.any(a[0]) for a in alone.values())


@pytest.mark.parametrize("count,n", [(5, 1024), (90, 512)])
def test_signal_reads_follow_the_last_solve(count, n):
    h = ga.ManyRHS(256, n, 12, count, "bf16", ga.options(tol=1e-6, seed=5, vecDistribution="gaussian"))
    h.solve()
    full = _check_reads(h, count, lambda r: r)
    [h.x(i) for i in range(count)]  # a window of the first solve is open
    h.configure(ref_outer=1, ref_inner=1, corrections=0)
    h.solve()
    short = [h.x(i)[0] for i in range(count)]
    alone = _check_reads(h, count, lambda r: r)
    for i in range(count):
        assert np.array_equal(short[i], alone[i][0])
    # vectors refined less differ from those refined in full, so a stale window would show
    assert any(not np.array_equal(short[i], full[i][0]) for i in range(count))


@pytest.mark.parametrize("ens,k,m,n,p", [("gen", 1, 3, 7, 0), ("gen", 30, 300, 2049, 0), ("dct", 500, 1 << 15, 1 << 17, 0),
                                         ("smv", 40, 3000, 65537, 7)])
def test_plan_errors_and_support_counts(ens, k, m, n, p):
    pl = ga.Plan("NIHT", ens, k, m, n, p, ga.options(tol=1e-6, seed=9, maxiter=20))
    pl.solve()
    r = pl.results()
    x, t = r["x"].astype(np.float64), r["x_true"].astype(np.float64)
    ref = [np.abs(t - x).sum() / np.abs(t).sum(), np.sqrt(((t - x) ** 2).sum()) / np.sqrt((t ** 2).sum()),
           np.abs(t - x).max() / np.abs(t).max()]
    # 64-bit sums rounded once to float32: half an ulp, and 2^-50 per sum for its order
    assert np.allclose(r["norms"], ref, rtol=2.0 ** -23, atol=0)
    tp = int(((t != 0) & (x != 0)).sum())
    tn = int(((t == 0) & (x == 0)).sum())
    assert list(r["support"]) == [tp, k - tp, tn, n - k - tn]
    pl.close()


@pytest.mark.parametrize("rows", [1, 32768, 32769])
def test_network_scores_with_and_without_staging(rows):
    net = ga.MLP(seed=2)
    X = np.abs(np.random.default_rng(1).standard_normal((rows, 8))).astype(np.float32)
    whole = net.scores(X)
    parts = np.concatenate([net.scores(X[i:i + 4096]) for i in range(0, rows, 4096)])
    assert np.array_equal(whole, parts)


def test_given_problems_from_more_threads_than_idle_lanes():
    rng = np.random.default_rng(4)
    probs = []
    for i in range(8):
        m, n, k = 64 + 8 * i, 200 + 31 * i, 5
        A = np.asfortranarray(rng.standard_normal((m, n)).astype(np.float32) / np.float32(np.sqrt(m)))
        x = np.zeros(n, np.float32)
        x[rng.choice(n, k, replace=False)] = 1
        probs.append((A @ x, A, k))
    call = lambda q: ga.cs("NIHT", "gen", *q, ga.options(tol=1e-6))[0]  # noqa: E731
    want = [call(q) for q in probs]
    got = [[None] * 3 for _ in probs]

    def work(i):
        for r in range(3):
            got[i][r] = call(probs[i])
    th = [threading.Thread(target=work, args=(i,)) for i in range(len(probs))]
    [t.start() for t in th]
    [t.join() for t in th]
    for i, q in enumerate(probs):
        assert all(np.array_equal(g, want[i]) for g in got[i]), i


@pytest.mark.parametrize("n", [1 << 12, 1 << 16, 1 << 17])  # with the staging memory, its last size, past it
def test_given_problem_solutions_of_every_length(n):
    from gaga_amd import _capi
    rng = np.random.default_rng(6)
    m, k = n // 4, n // 256
    rows = np.sort(rng.choice(n, m, replace=False)).astype(np.int32)
    x = np.zeros(n, np.float32)
    x[rng.choice(n, k, replace=False)] = rng.choice([-1.0, 1.0], k)
    y = _capi.apply("dct", 0, m, n, x, dct_rows=rows)
    got, iters, _ = ga.cs("NIHT", "dct", y, rows + 1, k, m, n, ga.options(tol=1e-5))
    # stops at |r| <= tol; the smallest singular value on 2k columns is above 1 / 4 here
    # (a quarter of the rows of an orthogonal matrix, scale 1 / 2)
    assert np.linalg.norm(got - x) <= 8e-5 and iters > 0
    assert set(np.flatnonzero(np.abs(got) > 0.5)) == set(np.flatnonzero(x))
