"""The 256 x 128 tile's pipeline at its ends: one, two, three and four K stages,
ragged column counts around a tile, through the kernel-level product (M = 256 mod
512 takes that tile), against float64 products of the quantized operands.  FP32
accumulation: |error| <= K 2^-23 sum |a||b|."""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("fmt,stage", [("bf16", 64), ("fp8", 128)])
@pytest.mark.parametrize("stages,N", [(1, 1), (2, 127), (3, 128), (4, 129), (7, 300)])
def test_tile_pipeline(lib, fmt, stage, stages, N):
    M, K = 768, stage * stages
    rng = np.random.default_rng(stages)
    A = rng.standard_normal((M, K)).astype(np.float32)
    B = rng.standard_normal((N, K)).astype(np.float32)
    C, Aq, Bq = lib.gemm_tn(fmt, A, B)
    Aq, Bq = Aq.astype(np.float64), Bq.astype(np.float64)
    assert (np.abs(C - Aq @ Bq.T) <= K * 2.0 ** -23 * (np.abs(Aq) @ np.abs(Bq).T) + 1e-30).all()
