"""GPU parity of the lm_head of several hidden states (batch_gemv.hip), where
its slices and tiles end: M around 4, 8, 16, 32 and past the rows of one
launch, N around a 16-row tile, the shortest and longest K.  The bound is the
one of tests/test_gpu_lmhead.py, 2^-16 sum_k |x_k w_k| per logit."""
import numpy as np
import pytest

from hachiue_amd import hip
from oracle import pyoracle as o
from tests.test_gpu_lmhead import FORMATS, check, run_gemv
from tests.test_oracle_lmhead import random_blocks

pytestmark = pytest.mark.gpu

BATCHED = ["q4_k", "q6_k"]


@pytest.mark.parametrize("fmt", BATCHED)
@pytest.mark.parametrize("M,K,N", [(2, 256, 16), (3, 512, 33), (4, 4096, 1000), (5, 256, 4099),
                                   (8, 1024, 17), (9, 768, 5000), (16, 512, 65), (17, 256, 4096),
                                   (32, 4096, 200), (33, 512, 999), (64, 1024, 3001),
                                   (259, 512, 40)])
def test_batched_rows(sampler, fmt, M, K, N):
    rng = np.random.default_rng(M * 1000 + K + N)
    w = random_blocks(FORMATS[fmt], N, K, rng)
    x = rng.standard_normal((M, K)).astype(np.float32)
    x[M // 2] *= np.exp2(rng.integers(-20, 20, K)).astype(np.float32)
    x[-1, ::3] = 0.0
    y = run_gemv(sampler, FORMATS[fmt], x, w, N, ldx=K + 4, ldy=N + 3)
    check(FORMATS[fmt], x, w, N, y)


@pytest.mark.parametrize("fmt", BATCHED)
def test_batched_rows_full_vocabulary(sampler, fmt):
    rng = np.random.default_rng(5)
    M, K, N = 20, 1024, 151936
    w = random_blocks(FORMATS[fmt], N, K, rng)
    x = rng.standard_normal((M, K)).astype(np.float32)
    y = run_gemv(sampler, FORMATS[fmt], x, w, N)
    check(FORMATS[fmt], x[[0, 7, 19]], w, N, y[[0, 7, 19]])
    # the same rows again, alone in their slice: a row's logits do not depend
    # on its neighbours
    again = run_gemv(sampler, FORMATS[fmt], x[17:], w, N)
    check(FORMATS[fmt], x[[19]], w, N, again[[2]])


@pytest.mark.parametrize("fmt", ["q4_k", "q6_k"])
@pytest.mark.parametrize("bad", [np.inf, -np.inf, np.nan])
def test_batched_row_with_non_finite_input(sampler, fmt, bad):
    """The row of a non-finite element is NaN everywhere, its neighbours are
    untouched."""
    rng = np.random.default_rng(9)
    M, K, N = 11, 512, 300
    w = random_blocks(FORMATS[fmt], N, K, rng)
    x = rng.standard_normal((M, K)).astype(np.float32)
    x[6, 300] = bad
    y = run_gemv(sampler, FORMATS[fmt], x, w, N)
    assert np.isnan(y[6]).all()
    keep = [r for r in range(M) if r != 6]
    check(FORMATS[fmt], x[keep], w, N, y[keep])
