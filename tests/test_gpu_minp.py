"""GPU parity of the one-pass min-p kernel (topK >= vocab with min-p): rows
it finishes itself, in whole rows and split over four workgroups, rows it
gives to the general path, and the edges between them.  Tokens, cutoffs and
counts against the oracle; a draw or top-p sum within 1e-6 of a boundary may
differ (tests/gpu_util.py)."""
import numpy as np
import pytest

from tests.gpu_util import run_gpu, run_oracle
from tests.test_gpu_large import _check

pytestmark = pytest.mark.gpu
INF = float("inf")


@pytest.fixture(params=["auto", "whole", "split4"])
def ctx(request, sampler, sampler_whole, sampler_split):
    return {"auto": sampler, "whole": sampler_whole, "split4": sampler_split}[request.param]


@pytest.mark.parametrize("vocab", [1028, 4100, 32767, 32772, 65541, 151936])
def test_options_and_sizes(ctx, vocab):
    rng = np.random.default_rng(vocab)
    stride = (vocab + 3) // 4 * 4
    cfgs = [dict(temperature=t, topK=INF, topP=p, minP=m)
            for t, p, m in [(1.0, 1.0, 0.05), (0.7, 0.9, 0.1), (1.5, 1.0, 0.004), (0.05, 1.0, 0.02),
                            (1.0, 0.3, 0.01), (1.0, 1.0, 1.0), (1.0, 1.0, 2.0), (30.0, 0.5, 0.5),
                            (1.0, 0.0, 0.05), (0.9, 0.95, 0.9)]]
    rows = len(cfgs)
    x = np.zeros((rows, stride), np.float32)
    x[:, :vocab] = rng.standard_normal((rows, vocab)) * 2.5
    for r in range(rows):
        x[r, rng.integers(0, vocab, 8)] += 12.0
    u = rng.random(rows)
    u[0], u[1] = 0.0, 1.0 - 2.0 ** -53
    hist = rng.integers(0, vocab, (rows, 40)).astype(np.int32)
    cfgs[3]["repetitionPenalty"] = 1.3
    cfgs[9].update(presencePenalty=0.4, frequencyPenalty=0.2)
    _check(ctx, x, vocab, hist.reshape(-1), np.arange(rows + 1, dtype=np.int64) * 40, cfgs, u, 64,
           f"min-p V={vocab}", want_cands=False)


def test_unusual_rows(ctx):
    """Masked rows, rows with no, one or two candidates, NaN, an infinite
    maximum, a maximum that only the last logits hold, more candidates than
    the list takes (finished by the general path), ties."""
    rng = np.random.default_rng(3)
    vocab, rows = 70002, 14
    x = np.full((rows, 70004), -np.inf, np.float32)
    base = (rng.standard_normal((rows, vocab)) * 2).astype(np.float32)
    x[1, 5] = -3.0                                   # one candidate
    x[2, [7, 69999]] = [1.0, 0.5]                    # two, far apart
    x[3, 40000:40050] = base[3, :50]                 # a grammar's few allowed ids
    x[4, :vocab] = base[4]
    x[4, ::3] = np.nan
    x[5, :vocab] = base[5]
    x[5, 123] = np.inf
    x[6, 9] = np.inf                                 # infinite and alone
    x[7, :vocab] = np.sort(base[7])                  # rises to the end
    x[8, :vocab] = 0.25                              # all equal: every logit is a candidate
    x[9, :vocab] = np.round(base[9])                 # ties among the candidates
    x[10, :vocab] = base[10]
    x[10, vocab - 1] = 60.0                          # the maximum past the last whole float4
    x[11, :vocab] = base[11] - 3e38 * (rng.random(vocab) < 0.5)
    x[12, :vocab] = -0.0
    x[12, 10:20] = 0.0
    x[13, :vocab] = base[13] * 1e-3                  # nearly flat: more than the list takes
    cfgs = [dict(temperature=1.0, topK=INF, topP=1.0, minP=0.05, ) for _ in range(rows)]
    cfgs[10]["temperature"] = 0.02
    u = rng.random(rows)
    _check(ctx, x, vocab, None, None, cfgs, u, 64, "min-p unusual rows", want_cands=False)


@pytest.mark.parametrize("vocab", [1025, 5003, 65538, 151939])
@pytest.mark.parametrize("opts", [dict(minP=0.02), dict(), dict(topK=3000, minP=0.02)])
def test_unaligned_rows(ctx, vocab, opts):
    """Odd strides: rows that start at any multiple of four bytes, on the
    min-p, two-pass and general kernels; then with candidate outputs (the
    general path)."""
    rng = np.random.default_rng(vocab)
    rows = 5
    x = (rng.standard_normal((rows, vocab)) * 2).astype(np.float32)
    cfgs = [dict(dict(temperature=1.0, topK=INF, topP=0.95), **opts)] * rows
    u = rng.random(rows)
    _check(ctx, x, vocab, None, None, cfgs, u, 64, "unaligned", want_cands=False)
    _check(ctx, x, vocab, None, None, cfgs, u, 64, "unaligned, candidates", want_cands=True)


def test_mixed_batch(ctx):
    """Min-p rows beside rows of every other route, twice (the counters are
    back at zero)."""
    rng = np.random.default_rng(6)
    vocab, rows = 40000, 12
    x = (rng.standard_normal((rows, vocab)) * 2.5).astype(np.float32)
    kinds = [dict(topK=INF, minP=0.05), dict(topK=40), dict(topK=500), dict(topK=INF, topP=0.9),
             dict(topK=3000, minP=0.1), dict(temperature=0.0)]
    cfgs = [dict(kinds[r % 6], repetitionPenalty=1.1 if r % 2 else 1.0) for r in range(rows)]
    hist = rng.integers(0, vocab, (rows, 30)).astype(np.int32)
    for _ in range(2):
        _check(ctx, x, vocab, hist.reshape(-1), np.arange(rows + 1, dtype=np.int64) * 30, cfgs,
               rng.random(rows), 64, "min-p mixed", want_cands=False)


def test_normaliser_of_a_heavy_tail(ctx):
    """Rows whose mass lies mostly in 600,000 equal logits far below the
    candidates, so that a weight's error does not average out, at a value
    where an exponent rounded to binary32 would be off by most of half a unit
    (up to 6e-7 of the weight), with a top-p 3e-7 above or below a cumulative
    probability: the cutoff and the token are the oracle's.  (Weights within
    2^-23, the probabilities' own rounding 2^-24: below the 3e-7.)"""
    rng = np.random.default_rng(17)
    rows, vocab = 24, 600003
    x = np.zeros((rows, vocab), np.float32)
    cfgs, u, cuts = [], [], []
    for r in range(rows):
        t = float(rng.uniform(0.5, 1.3))
        top = np.float32(rng.uniform(7.0, 9.0))
        tail = np.float32(0)
        while True:
            tail = np.float32(top - t * rng.uniform(11.2, 12.0))
            y = float(np.float32(tail - top)) / t / np.log(2.0)
            off = (float(np.float32(y)) - y) * np.log(2.0)
            if abs(off) > 5e-7:
                break
        x[r] = tail
        near = rng.choice(vocab, 6, replace=False)
        x[r, near] = top - (t * np.array([0.0, 4.0, 4.2, 4.4, 4.6, 4.8])).astype(np.float32)
        e = np.exp((x[r].astype(np.float64) - float(top)) / t).astype(np.float32).astype(np.float64)
        p = (e[near] / e.sum()).astype(np.float32).astype(np.float64)
        j = int(rng.integers(0, 5))
        up = int(off < 0)         # where the rounded exponent is too small, so is the sum
        c = np.cumsum(p)[j] * (1 + (3e-7 if up else -3e-7))
        cfgs.append(dict(temperature=t, topK=INF, topP=c, minP=0.006))
        cuts.append(j + 1 + up)
        u.append(rng.uniform(0.02, 0.6))
    got = run_gpu(ctx, x, vocab, None, None, cfgs, np.array(u), 64, want_cands=False)
    want, _ = run_oracle(x, vocab, None, None, cfgs, np.array(u), 64)
    assert want.cutoff.tolist() == cuts
    assert got.cutoff.tolist() == cuts
    assert got.tokens.tolist() == want.token.tolist()


def test_rows_handed_to_the_general_path(ctx):
    """More candidates than the kernel sorts: the general path starts from the
    extremes and the count found here, also where they come from a row whose
    list was full early, with -Infinity and NaN among the logits, all above or
    all below zero, and a maximum or minimum past the last whole float4."""
    rng = np.random.default_rng(31)
    rows, vocab = 10, 120003
    x = (rng.standard_normal((rows, vocab)) * 0.7).astype(np.float32)
    x[1, ::2] = -np.inf
    x[2, ::3] = np.nan
    x[3] += 15.0
    x[4] -= 15.0
    x[5, -1] = x[5].max() + 0.5
    x[6, -1] = -40.0
    x[7, 60000:] = -np.inf                              # whole parts without a logit
    x[8] = np.round(x[8] * 4) / 4
    x[9, 0], x[9, -1] = 3.4e38, -3.4e38
    cfgs = [dict(temperature=1.0, topK=INF, topP=p, minP=m) for p, m in
            [(1.0, 0.02), (0.9, 0.05), (1.0, 0.1), (0.8, 0.02), (1.0, 0.02), (1.0, 0.03), (0.5, 0.02),
             (1.0, 0.02), (0.7, 0.02), (0.9, 0.05)]]
    cfgs[9]["temperature"] = 1e38
    _check(ctx, x, vocab, None, None, cfgs, rng.random(rows), 64, "min-p, handed over", want_cands=False)


def test_small_temperatures(ctx):
    """Temperatures whose reciprocal overflows a binary32 or a binary64."""
    rng = np.random.default_rng(23)
    vocab = 9001
    temps = [1e-6, 1e-20, 1e-37, 1e-39, 1e-300, 1e-310, 5e-324, 1e6, 1e38, 1e300]
    x = (rng.standard_normal((len(temps), vocab)) * 3).astype(np.float32)
    x[:, 77] = x[:, 4000] = 20.0
    cfgs = [dict(temperature=t, topK=INF, topP=0.9, minP=0.1) for t in temps]
    _check(ctx, x, vocab, None, None, cfgs, rng.random(len(temps)), 64, "min-p temperatures",
           want_cands=False)
