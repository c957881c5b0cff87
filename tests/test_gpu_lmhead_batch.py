"""GPU parity of the lm_head of several hidden states (batch_gemv.hip), where
its slices and tiles end: M around 4, 8, 16, 32 and past the rows of one
launch, N around a 16-row tile, the shortest and longest K, within the bound
of tests/test_gpu_lmhead.py, 2^-16 sum_k |x_k w_k| per logit.  Then what that
bound does not see: the accuracy against a row at a time, and rows that are
not finite."""
import ctypes

import numpy as np
import pytest

from hachiue_amd import Sampler, hip
from hachiue_amd import sampler as hsamp
from oracle import pyoracle as o
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


def batched_n(fmt, M, K):
    """Weight rows from which on M rows go together (gemv_batched)."""
    n = {"q4_k": (240000 if M > 8 else 131072) / M, "q6_k": (160000 if M > 8 else 120000) / M,
         "q1_0": 90e6 / K if M == 2 else 10000 / M, "ptq1_0": 32000 if M == 3 else 20000 / M,
         "q4_0": 12288 / M, "f32": (24576 if M < 16 else 16000) / M}
    n["pq2_0"], n["q4_1"] = n["q1_0"], n["q4_0"]
    return max(256, int(np.ceil(n[fmt])))


@pytest.mark.parametrize("fmt", list(ALL))
@pytest.mark.parametrize("M,K,extra", [(2, 1, 0), (3, 2, 1), (4, 0, 15), (5, 1, 16), (8, 4, 17), (9, 3, 5),
                                       (16, 2, 33), (17, 1, 8), (32, 0, 3), (33, 2, 31), (64, 3, 7),
                                       (259, 1, 2)])
def test_rows_taken_together(sampler, fmt, M, K, extra):
    """The batched kernels at the edges of their slices and of the rule that
    takes them: from its least number of weight rows on, the last tile ragged
    by `extra`.  Checked on the first, the last and some other weight rows."""
    if M < {"ptq1_0": 3, "q4_0": 4, "q4_1": 4, "f32": 4}.get(fmt, 2):
        pytest.skip("a row at a time")
    K = K * STEP.get(fmt, 512) or 4096
    N = batched_n(fmt, M, K) + extra
    rng = np.random.default_rng(M * 1000 + K + extra)
    w = random_blocks(ALL[fmt], N, K, rng)
    x = rng.standard_normal((M, K)).astype(np.float32)
    x[M // 2] *= np.exp2(rng.integers(-20, 20, K)).astype(np.float32)
    x[-1, ::3] = 0.0
    y = run(sampler, fmt, x, w, N, pad=3)
    rows = np.unique(np.concatenate([np.arange(40), np.arange(N - 40, N), rng.integers(0, N, 200)]))
    check(ALL[fmt], x, w[rows], len(rows), y[:, rows])


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
    M, K, N = 11, 512, 22003
    w = random_blocks(ALL[fmt], N, K, rng)
    x = rng.standard_normal((M, K)).astype(np.float32)
    x[6, 40] = bad                                  # (slabs follow it)
    x[9, [3, 400]] = bad                            # both signs of it, by the weights
    y = run(sampler, fmt, x, w, N)
    for r in (6, 9):
        alone = run(sampler, fmt, x[[r]], w, N)[0]
        assert not np.isfinite(alone).any()
        assert np.array_equal(y[r], alone, equal_nan=True), (r, y[r, :8], alone[:8])
        if fmt not in ("f32", "q4_1"):
            assert np.isnan(y[r]).all()
    keep = [r for r in range(M) if r not in (6, 9)]
    check(ALL[fmt], x[keep], w, N, y[keep])


def test_batched_f32_sums_that_overflow(sampler):
    """Finite inputs whose products or partial sums pass the largest binary32:
    an infinity stays one through the slabs after it, as in a call of one row."""
    rng = np.random.default_rng(10)
    M, K, N = 5, 512, 5003
    w = rng.standard_normal((N, K)).astype(np.float32)
    w[:, 5] = np.where(np.arange(N) % 2, 8.0, -8.0)
    x = rng.standard_normal((M, K)).astype(np.float32)
    x[2, 5] = 3e38
    y = run(sampler, "f32", x, w.view(np.uint8), N)
    assert np.array_equal(y[2], np.where(np.arange(N) % 2, np.inf, -np.inf).astype(np.float32))
    assert np.isfinite(y[[0, 1, 3, 4]]).all()


# ---- accuracy: no coarser than a row at a time

def without_channels(fmt, w, K, cols):
    """The weights of the given channels set to 0 (of their sub-blocks too,
    where a minimum is shared)."""
    if fmt == "f32":
        v = w.view(np.float32).reshape(-1, K).copy()
        v[:, cols] = 0.0
        return v.view(np.uint8)
    B, BB = o.block_spec(ALL[fmt])
    w = w.reshape(w.shape[0], K // B, BB).copy()
    for c in cols:
        blk, p = w[:, c // B], c % B          # (a view: written in place)
        if fmt in ("q4_0", "q4_1"):           # q = 8; Q4_1's minimum is -8 d
            i, hi = (2 if fmt == "q4_0" else 4) + p % 16, p >= 16
            blk[:, i] = (blk[:, i] & 0x0F) | 0x80 if hi else (blk[:, i] & 0xF0) | 8
            if fmt == "q4_1":
                d = blk[:, 0:2].copy().view(np.float16)
                blk[:, 2:4] = (d * np.float16(-8)).view(np.uint8)
        elif fmt == "q4_k":                   # q = 0 and no minima in the super-block
            i, hi = 16 + 32 * (p // 64) + p % 32, p % 64 >= 32
            blk[:, i] &= 0x0F if hi else 0xF0
            blk[:, 2:4] = 0
        else:                                 # q6_k: q = 32
            n, quarter, pos = p // 128, p % 128 // 32, p % 32
            i, h = 64 * n + 32 * (quarter & 1) + pos, 128 + 32 * n + pos
            blk[:, i] &= 0x0F if quarter >= 2 else 0xF0
            blk[:, h] = (blk[:, h] & ~np.uint8(3 << 2 * quarter)) | np.uint8(2 << 2 * quarter)
    return w.reshape(w.shape[0], -1)


def error(fmt, x, w, N, y):
    """Per row: rms error against binary64 over the logits' rms."""
    exact, _ = o.gemv_exact(ALL[fmt], x, w, N)
    e = y.astype(np.float64) - exact
    return np.sqrt((e ** 2).mean(-1) / (exact ** 2).mean(-1))


@pytest.mark.parametrize("fmt,outlier", [(f, s) for f in FORMATS for s in (1.0, 10.0, 1e3, 1e5, 1e8, 1e15)]
                         + [(f, 1.0) for f in PLANAR])
def test_batched_accuracy_with_outlier_channels(sampler, fmt, outlier):
    """Hidden states with outlier channels whose weights are 0, so that all of
    the signal lies in the small elements: the error against binary64 is not
    above a row's own.  (Both are sums of binary32 values over 2048 products;
    1.25 and 2^-24 allow for the order of their roundings.  A lost last limb
    would be an error of 2^-20 without outliers.)  The planar formats hold x as
    a row alone does."""
    rng = np.random.default_rng(int(np.log10(outlier)) + 3)
    M, K = 20, 2048
    N = max(batched_n(fmt, m, K) for m in (20, 7, 4, 3, 2))
    sub = rng.choice(N, 1500, replace=False)      # the weight rows looked at
    cols = [37, 700, 1301, 1999]
    w = random_blocks(ALL[fmt], N, K, rng)
    if fmt in FORMATS:
        w = without_channels(fmt, w, K, cols)
    x = rng.standard_normal((M, K)).astype(np.float32)
    x[:, cols] = (np.sign(x[:, cols]) * (0.5 + rng.random((M, len(cols)))) * outlier).astype(np.float32)
    rows = np.array([0, 1, 2, 3, 6, 11, 19])
    alone = [run(sampler, fmt, x[[r]], w, N)[:, sub] for r in rows]
    one = np.concatenate([error(fmt, x[[r]], w[sub], 1500, y) for r, y in zip(rows, alone)])
    least = {"ptq1_0": 3, "q4_0": 4, "q4_1": 4, "f32": 4}.get(fmt, 2)
    for m in (M, 7, 4, 3, 2):
        y = run(sampler, fmt, x[:m], w, N)[:, sub]
        # together or a row at a time, as the rule has it
        assert np.array_equal(y[0], alone[0][0]) == (m < least), m
        e = error(fmt, x[:m], w[sub], 1500, y)[rows[rows < m]]
        ref = one[rows < m]
        print(f"[accuracy] {fmt} outlier {outlier:g} M {m}: {e.mean():.2e}, one row {ref.mean():.2e}", flush=True)
        assert (e <= 1.25 * ref + 2.0 ** -24).all(), (m, e, ref)


@pytest.mark.parametrize("fmt", ["q4_k", "q6_k"])
def test_batched_outliers_near_the_binary32_range(sampler, fmt):
    """Channels near the largest binary32 with weights of 0, block scales near
    the largest binary16: the scale times the limbs' unit passes the range, no logit does,
    here as in a row alone."""
    rng = np.random.default_rng(21)
    M, K = 6, 1024
    N = batched_n(fmt, M, K)
    cols = [9, 300, 1000]
    w = without_channels(fmt, random_blocks(ALL[fmt], N, K, rng, scale=2e4), K, cols)
    x = rng.standard_normal((M, K)).astype(np.float32)
    x[1::2, cols] = 5e36
    y = run(sampler, fmt, x, w, N)
    sub = rng.choice(N, 300, replace=False)
    for r in range(M):
        alone = run(sampler, fmt, x[[r]], w, N)[0]
        assert np.isfinite(alone).all() and np.isfinite(y[r]).all(), r
        # (the groups of the huge channels lose their other elements, alone too)
        if r % 2 == 0:
            check(ALL[fmt], x[[r]], w[sub], 300, y[[r]][:, sub])


# ---- graphs

@pytest.mark.parametrize("fmt", ["q6_k", "pq2_0", "f32"])
def test_first_call_captured(sampler, fmt):
    """A context whose first batched call is being captured: the graph holds
    the batched kernels, and each replay, with eager calls between, gives the
    eager call's results bit for bit."""
    R = hip.runtime()
    vp = ctypes.c_void_p
    R.hipStreamBeginCapture.argtypes = [vp, ctypes.c_int]
    R.hipStreamEndCapture.argtypes = [vp, ctypes.POINTER(vp)]
    R.hipGraphInstantiate.argtypes = [ctypes.POINTER(vp), vp, vp, vp, ctypes.c_size_t]
    R.hipGraphLaunch.argtypes = [vp, vp]
    R.hipGraphExecDestroy.argtypes = R.hipGraphDestroy.argtypes = [vp]
    rng = np.random.default_rng(8)
    M, K, N = 9, 1024, 17800
    w = random_blocks(ALL[fmt], N, K, rng)
    xs = [rng.standard_normal((M, K)).astype(np.float32) for _ in range(3)]
    want = [run(sampler, fmt, x, w, N) for x in xs]
    if fmt in PLANAR:
        q, sc = hsamp.split_blocks(ALL[fmt], w)
        d_w, d_s = hip.DeviceArray.from_numpy(q), hip.DeviceArray.from_numpy(sc)
    else:
        d_w, d_s = hip.DeviceArray.from_numpy(np.ascontiguousarray(w).reshape(-1)), None
    wt = hsamp.weights(ALL[fmt], N, K, d_w.addr, d_s.addr if d_s else None, False, None)
    d_x, d_y = hip.DeviceArray.from_numpy(xs[0]), hip.DeviceArray((M, N), np.float32)
    d_y2 = hip.DeviceArray((M, N), np.float32)
    st, graph, ex = hip.Stream(), vp(), vp()
    print(f"[gpu] captured batched lm_head {fmt}", flush=True)
    with Sampler(0) as ctx:
        hip.check(R.hipStreamBeginCapture(st.handle, 0), "hipStreamBeginCapture")   # global mode
        try:
            ctx.gemv_device_ex(d_x.addr, M, K, wt, d_y.addr, N, stream=st)
        finally:
            hip.check(R.hipStreamEndCapture(st.handle, ctypes.byref(graph)), "hipStreamEndCapture")
        hip.check(R.hipGraphInstantiate(ctypes.byref(ex), graph, None, None, 0), "hipGraphInstantiate")
        for x, y in zip(xs, want):
            d_x.upload(x)
            d_y.upload(np.zeros((M, N), np.float32))
            hip.synchronize()
            hip.check(R.hipGraphLaunch(ex, st.handle), "hipGraphLaunch")
            st.synchronize()
            assert np.array_equal(d_y.download().view(np.uint32), y.view(np.uint32))
            ctx.gemv_device_ex(d_x.addr, M, K, wt, d_y2.addr, N, stream=st)
            st.synchronize()
            assert np.array_equal(d_y2.download().view(np.uint32), y.view(np.uint32))
        R.hipGraphExecDestroy(ex)
        R.hipGraphDestroy(graph)
    st.destroy()
