"""Waits that are bounded by a tiny limit end every form of a solve with an error
instead of results: the general form's barriers on a team (an algorithm that the
LDS forms do not take), the split form with and without its extra hop for a
histogram in memory, and teams of a batch with instances of unlike lengths, whose
support lists then stay within each instance.  With the default bound the same
solves succeed."""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu

TOL = 1e-5


@pytest.mark.parametrize("mode", ["device", "plain"])
@pytest.mark.parametrize("alg,ens,k,m,n,p,extra", [
    ("FIHT", "gen", 100, 2048, 8192, 0, {"teamSize": 16}),
    ("FIHT", "dct", 60, 4001, 16384, 0, {"teamSize": 16}),
    ("NIHT", "smv", 60, 2000, 8191, 7, {"teamSize": 16, "numBins": 5000}),
    ("CGIHT", "smv", 60, 4000, 20000, 7, {"teamSize": 64}),
    ("HTP", "dct", 60, 4001, 16384, 0, {"teamSize": 16}),
])
def test_plans(lib, mode, alg, ens, k, m, n, p, extra):
    kw = dict(extra, tol=TOL, seed=20260101, mode=mode)
    if ens == "smv":
        kw["matrixEnsemble"] = "binary"
    pl = lib.Plan(alg, ens, k, m, n, p, lib.options(barrierSpinLimit=1, **kw))
    assert pl.form()[0] == ("general" if alg == "FIHT" else "split")
    for _ in range(2):
        with pytest.raises(lib.GagaError, match="team barrier timed out"):
            pl.solve()
    pl.close()
    pl = lib.Plan(alg, ens, k, m, n, p, lib.options(**kw))
    pl.solve()
    r = pl.results()
    pl.close()
    assert r["stop_reason"] == 0 and r["norms"][2] < 1e-4


@pytest.mark.parametrize("cfg", [(4, 512, -1), (4, 512, 8), (16, 512, 20)])
def test_batch_teams(lib, cfg):
    specs = []
    for i in range(24):  # the largest come first in the queue: a team goes on to shorter ones
        n = (4096, 1024, 512)[i % 3]
        specs.append(dict(ens="smv" if i % 4 == 3 else "gen", k=12, m=n // 4, n=n, p=7, instance=i))
    for limit in (1, 0):
        B = lib.Batch("CGIHT", specs, lib.options(tol=TOL, seed=20260101, blockSize=512, barrierSpinLimit=limit))
        B.configure(*cfg)
        if limit:
            for _ in range(2):
                with pytest.raises(lib.GagaError, match="team barrier timed out"):
                    B.solve()
        else:
            B.solve()
            assert (B.results()["stop_reason"] == 0).mean() > 0.9
            assert np.median(B.results()["norms"][:, 2]) < 1e-4
        B.close()
