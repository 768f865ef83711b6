"""Batches whose teams are enlarged where the chip has room (every instance
beside the teams, the small ones after them, nothing but teams, a team size that
is no power of two), against the same batch one workgroup per instance; the
configured geometry is what the batch reports."""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu

TOL = 1e-5


@pytest.mark.parametrize("alg", ["NIHT", "CGIHT"])
@pytest.mark.parametrize("count,team,big", [(1, 4, 1), (6, 4, 2), (6, 3, 6), (70, 4, 65), (300, 2, 4)])
def test_enlarged_teams(lib, alg, count, team, big):
    specs = []
    for i in range(count):
        if i < big:  # 16.8 and 4.2 MB a product: teams grow for the first
            n = 4096 if i == 0 else 2048
            specs.append(dict(ens="gen", k=20, m=n // 4, n=n, instance=i))
        else:
            specs.append(dict(ens="smv" if i % 2 else "gen", k=6, m=120 + i % 3, n=400, p=7, instance=i))
    B = lib.Batch(alg, specs, lib.options(tol=TOL, seed=20260101, blockSize=512))
    out = []
    for cfg in ((team, 512, big), (1, 512, 0)):
        B.configure(*cfg)
        B.solve()
        r = B.results()
        xs = [B.x(i) for i in range(count)]
        B.solve()
        assert all(np.array_equal(B.x(i)[0], xs[i][0]) for i in range(count))
        assert B.info()["team_size"] == cfg[0]
        out.append((r, xs))
    (a, xa), (b, xb) = out
    assert np.abs(a["iters"] - b["iters"]).max() <= 1
    for i in range(count):
        # both stop at |r| <= tol: |x - x_true| <= tol / sigma with the smallest singular
        # value on 2k columns above 1 / 3 at these densities
        if a["stop_reason"][i] == 0 and b["stop_reason"][i] == 0:
            assert np.linalg.norm(xa[i][0] - xb[i][0]) <= 6 * TOL
    assert (a["stop_reason"] == b["stop_reason"]).all()
