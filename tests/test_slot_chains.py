"""The rule by which the mid kernel settles a draw inside a group of equal
logits (src/sampler.ts:50-74): a logit that enters the k slots takes the slot
of the smallest of the k largest before it, back to one of the first k, whose
slot is its index.  Restated here and checked against the oracle's scan (CPU),
then the kernel itself on rows whose draw falls in such a group (GPU)."""
import numpy as np
import pytest

from oracle import pyoracle as o


def chain_slot(row, k, idx):
    """Slot of the logit at idx, which enters; None where a leaving value
    is not unique in its prefix."""
    while idx >= k:
        before = row[:idx]
        m = np.partition(before, idx - k)[idx - k]      # the k-th largest
        where = np.flatnonzero(before == m)
        if where.size != 1:
            return None
        idx = int(where[0])
    return idx


@pytest.mark.parametrize("k", [2, 5, 65, 300])
@pytest.mark.parametrize("V", [301, 2000, 20000])
def test_chains_give_the_scans_order(k, V):
    if k >= V:
        pytest.skip("every logit keeps its slot")
    rng = np.random.default_rng(k * 7 + V)
    settled = 0
    for trial in range(6):
        row = rng.standard_normal(V).astype(np.float32)
        top = np.argsort(-row)[:k]
        for _ in range(1 + k // 20):                    # equal values among the k largest
            a, b = rng.choice(top, 2, replace=False)
            row[a] = row[b]
        if trial == 5:
            row = np.round(row * 200).astype(np.float32) / 200   # ties everywhere
        res = o.sample_batch(row[None].copy(), V, None, None,
                             [dict(temperature=1.0, topK=k, topP=1.0)], np.array([0.5]), o.HEAP, k)
        ids = res.cand_ids[0, :k]
        vals = row[ids]
        kth = vals[-1]
        i = 0
        while i < k:
            j = i + 1
            while j < k and vals[j] == vals[i]:
                j += 1
            if j - i > 1 and vals[i] > kth:
                slots = [chain_slot(row, k, int(x)) for x in ids[i:j]]
                if None not in slots:
                    assert slots == sorted(slots)
                    settled += 1
            i = j
    assert settled > 0 or k == 2     # (two slots hold no group above the k-th)


@pytest.mark.gpu
@pytest.mark.parametrize("k,V", [(65, 70), (70, 4097), (100, 262144), (300, 151936), (640, 60001),
                                 (1000, 151936), (1024, 400000), (1024, 1030)])
def test_draws_inside_equal_values(sampler, k, V):
    from tests.gpu_util import compare, run_gpu, run_oracle
    rng = np.random.default_rng(k + V)
    rows = 16
    x = (rng.standard_normal((rows, V)) * 2).astype(np.float32)
    for r in range(rows):
        top = np.argsort(-x[r])[:k]
        # the largest value several times, at random places, so that the draw
        # falls among them
        n = 2 + r % 4 if r < 12 else 40
        n = min(n, k - 2)
        where = rng.choice(V, n, replace=False)
        x[r, where] = x[r, top[0]] + 1.0
        if r == 10:
            x[r, 3] = -np.inf                 # the first k are not all finite
        if r == 11:
            x[r] = np.round(x[r] * 4) / 4     # leaving values that are not unique
    cfgs = [dict(temperature=0.3, topK=k, topP=1.0)] * rows
    u = rng.random(rows) * 0.9
    for stride in (V, V + 1):
        y = np.zeros((rows, stride), np.float32)
        y[:, :V] = x
        got = run_gpu(sampler, y, V, None, None, cfgs, u, 64, stride=stride, want_cands=False)
        want, ref = run_oracle(y, V, None, None, cfgs, u, 64)
        compare(got, want, ref, cfgs, V, 64, f"equal values k={k} V={V}")
        assert (got.flags & 0x2).any()
