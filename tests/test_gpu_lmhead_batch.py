"""GPU parity of the lm_head of several hidden states (batch_gemv.hip), where
its slices and tiles end: M around 4, 8, 16, 32 and past the rows of one
launch, N around a 16-row tile, the shortest and longest K, within the bound
of tests/test_gpu_lmhead.py, 2^-16 sum_k |x_k w_k| per logit.  Then rows that
are not finite."""
import numpy as np
import pytest

from tests.test_gpu_lmhead import FORMATS, PLANAR, check, run_gemv, run_gemv_ex
from tests.test_oracle_lmhead import random_blocks

pytestmark = pytest.mark.gpu

ALL = dict(FORMATS, **PLANAR)
STEP = {"f32": 64, "q4_0": 256, "q4_1": 256, "q4_k": 256, "q6_k": 256}   # of K; planar 512


def run(sampler, fmt, x, w, N, pad=0):
    if fmt in PLANAR:
        return run_gemv_ex(sampler, ALL[fmt], x, w, N, ldx=x.shape[1] + pad, ldy=N + pad)
    return run_gemv(sampler, ALL[fmt], x, w, N, ldx=x.shape[1] + pad, ldy=N + pad)


@pytest.mark.parametrize("fmt", list(ALL))
@pytest.mark.parametrize("M,K,N", [(2, 1, 16), (3, 2, 33), (4, 0, 1000), (5, 1, 4099),
                                   (8, 4, 17), (9, 3, 5000), (16, 2, 65), (17, 1, 4096),
                                   (32, 0, 200), (33, 2, 999), (64, 3, 3001), (259, 1, 40)])
def test_batched_rows(sampler, fmt, M, K, N):
    """K in steps of the format's slab (0: the longest, 4096)."""
    K = K * STEP.get(fmt, 512) or 4096
    rng = np.random.default_rng(M * 1000 + K + N)
    w = random_blocks(ALL[fmt], N, K, rng)
    x = rng.standard_normal((M, K)).astype(np.float32)
    x[M // 2] *= np.exp2(rng.integers(-20, 20, K)).astype(np.float32)
    x[-1, ::3] = 0.0
    y = run(sampler, fmt, x, w, N, pad=3)
    check(ALL[fmt], x, w, N, y)


@pytest.mark.parametrize("fmt", list(ALL))
def test_batched_rows_full_vocabulary(sampler, fmt):
    rng = np.random.default_rng(5)
    M, K, N = 20, 512 if fmt == "f32" else 1024, 151936
    w = random_blocks(ALL[fmt], N, K, rng)
    x = rng.standard_normal((M, K)).astype(np.float32)
    y = run(sampler, fmt, x, w, N)
    check(ALL[fmt], x[[0, 7, 19]], w, N, y[[0, 7, 19]])
    # some of the rows again, in a smaller batch
    again = run(sampler, fmt, x[13:], w, N)
    check(ALL[fmt], x[[19]], w, N, again[[6]])


@pytest.mark.parametrize("fmt", list(ALL))
@pytest.mark.parametrize("bad", [np.inf, -np.inf, np.nan])
def test_batched_row_with_non_finite_input(sampler, fmt, bad):
    """The row of a non-finite element is what it is in a call of its own, NaN
    or an infinity in the same places (NaN everywhere on the integer formats);
    its neighbours are untouched."""
    rng = np.random.default_rng(9)
    M, K, N = 11, 512, 300
    w = random_blocks(ALL[fmt], N, K, rng)
    x = rng.standard_normal((M, K)).astype(np.float32)
    x[6, 40] = bad                                  # (slabs follow it)
    x[9, [3, 400]] = bad                            # both signs of it, by the weights
    y = run(sampler, fmt, x, w, N)
    for r in (6, 9):
        alone = run(sampler, fmt, x[[r]], w, N)[0]
        assert not np.isfinite(alone).any()
        if fmt != "q4_1":
            assert np.array_equal(y[r], alone, equal_nan=True), (r, y[r, :8], alone[:8])
        if fmt not in ("f32", "q4_1"):
            assert np.isnan(y[r]).all()
    keep = [r for r in range(M) if r not in (6, 9)]
    check(ALL[fmt], x[keep], w, N, y[keep])


def test_batched_f32_sums_that_overflow(sampler):
    """Finite inputs whose products or partial sums pass the largest binary32:
    an infinity stays one through the slabs after it, as in a call of one row."""
    rng = np.random.default_rng(10)
    M, K, N = 5, 512, 200
    w = rng.standard_normal((N, K)).astype(np.float32)
    w[:, 5] = np.where(np.arange(N) % 2, 8.0, -8.0)
    x = rng.standard_normal((M, K)).astype(np.float32)
    x[2, 5] = 3e38
    y = run(sampler, "f32", x, w.view(np.uint8), N)
    assert np.array_equal(y[2], np.where(np.arange(N) % 2, np.inf, -np.inf).astype(np.float32))
    assert np.isfinite(y[[0, 1, 3, 4]]).all()
