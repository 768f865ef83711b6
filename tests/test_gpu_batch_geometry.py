"""The teams a batch runs in: what the solve launched is reported beside the
configured geometry, every large instance has its team at once where the chip has
room, exact teams on request, and the autotuner's choice solves the batch."""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu

TOL = 1e-5


def _same(B, want):
    B.solve()
    r = B.results()
    assert (r["stop_reason"] == want["stop_reason"]).all()
    assert np.abs(r["iters"] - want["iters"]).max() <= 1
    return r


def test_configured_and_run_geometry(lib):
    specs = [dict(ens="gen", k=20, m=512, n=2048, instance=i) for i in range(65)]
    specs += [dict(ens="gen", k=6, m=120, n=400, instance=i) for i in range(65, 70)]
    B = lib.Batch("CGIHT", specs, lib.options(tol=TOL, seed=20260101, blockSize=512))
    with pytest.raises(lib.GagaError, match="not been solved"):
        B.ran()
    B.solve()
    want = B.results()
    B.configure(4, 512, 65)  # 4.2 MB a product: no larger teams; 65 of them are 9 groups of eight
    _same(B, want)
    teams, size = B.ran()
    assert size == 4 and teams >= 65 and teams % 8 == 0
    B.close()


def test_exact_teams(lib):
    specs = [dict(ens="gen", k=50, m=1024, n=4096, instance=i) for i in range(6)]  # 16.8 MB a product
    B = lib.Batch("NIHT", specs, lib.options(tol=TOL, seed=20260101, blockSize=512))
    B.solve()
    want = B.results()
    B.configure(4, 512)
    _same(B, want)
    assert B.ran()[1] > 4 and B.info()["team_size"] == 4
    B.configure(4, 512, exact=True)
    _same(B, want)
    assert B.ran() == (6, 4)
    B.configure(4, 512)
    _same(B, want)
    assert B.ran()[1] > 4
    team, block, big, ms = B.tune(probe_iters=3)
    assert team in (1, 2, 4, 8) and block in (256, 512, 1024) and ms > 0
    _same(B, want)
    assert B.ran()[1] % team == 0
    B.close()
