"""The rule by which the mid kernel settles a draw inside a group of equal
logits (src/sampler.ts:50-74): a logit that enters the k slots takes the slot
of the smallest of the k largest before it, back to one of the first k, whose
slot is its index.  Restated here and checked against the oracle's scan (CPU),
with the kernel's limit on a group's members, then the kernel itself on rows
whose draw falls in such a group (GPU)."""
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


MEMBERS = 16     # the largest group settled by chains (kChaseMembers)


def chain_pick(row, k, ids, pick):
    """The kernel's answer for the draw at position `pick` of the candidates
    `ids` (value descending, index ascending): its scan for the group's ends
    stops one past the limit, and a group that may go on is not settled."""
    lo, hi = pick, pick + 1
    while lo > 0 and pick - lo < MEMBERS and row[ids[lo - 1]] == row[ids[pick]]:
        lo -= 1
    while hi < len(ids) and hi - pick <= MEMBERS and row[ids[hi]] == row[ids[pick]]:
        hi += 1
    if hi - lo > MEMBERS:
        return None
    slots = [chain_slot(row, k, int(x)) for x in ids[lo:hi]]
    return None if None in slots else int(ids[lo + np.argsort(slots)[pick - lo]])


def group_row(rng, V, n, first, k):
    """A row whose maximum occurs n times, `first` of them among the first k."""
    row = (rng.standard_normal(V) * 2).astype(np.float32)
    where = np.concatenate([rng.choice(k, first, replace=False),
                            k + rng.choice(V - k, n - first, replace=False)])
    row[where] = row.max() + np.float32(1.0)
    return row


@pytest.mark.parametrize("n", [2, 15, 16, 17, 18, 33])
def test_members_at_the_limit(n):
    """A group at, below and above the limit: the drawn member is the scan's,
    or the group is left to the scan; up to the limit it is settled."""
    rng = np.random.default_rng(n)
    k, V = 100, 4097
    for trial in range(8):
        row = group_row(rng, V, n, trial % min(n + 1, 4), k)
        res = o.sample_batch(row[None].copy(), V, None, None,
                             [dict(temperature=1.0, topK=k, topP=1.0)], np.array([0.5]), o.HEAP, k)
        ids = np.lexsort((np.arange(V), -row))[:k]
        for pick in {0, 1, 15, 16, n - 1} & set(range(n)):
            got = chain_pick(row, k, ids, pick)
            assert got is None if n > MEMBERS else got == res.cand_ids[0, pick], (trial, pick)


@pytest.mark.gpu
@pytest.mark.parametrize("n", [15, 16, 17, 18, 33])
@pytest.mark.parametrize("k,V", [(100, 4097), (700, 60001)])
def test_draws_at_the_member_limit(sampler, n, k, V):
    """Draws of the first, second, 16th, 17th and last member of a group at
    and above the limit, its members inside and outside the first k."""
    from tests.gpu_util import run_gpu, run_oracle
    rng = np.random.default_rng(n * 1000 + k)
    picks = [p for p in (0, 1, 15, 16, n - 1) if p < n]
    rows = 8 * len(picks)
    x = np.stack([group_row(rng, V, n, r // len(picks) % 4, k) for r in range(rows)])
    u = np.array([0.0 if picks[r % len(picks)] == 0 else (picks[r % len(picks)] + 0.5) / n
                  for r in range(rows)])
    cfgs = [dict(temperature=0.03, topK=k, topP=1.0)] * rows   # the others weigh nothing
    got = run_gpu(sampler, x, V, None, None, cfgs, u, 64, want_cands=False)
    want, _ = run_oracle(x, V, None, None, cfgs, u, 64)
    assert got.tokens.tolist() == want.token.tolist()


@pytest.mark.gpu
def test_draws_inside_equal_values_of_penalised_rows(sampler):
    """Penalties rewrite logits of the row in place, members of the group and
    logits of its chains among them; then the same through a decode step."""
    from hachiue_amd import hip
    from hachiue_amd.decode import DecodeState
    from tests.gpu_util import compare, run_gpu, run_oracle
    rng = np.random.default_rng(12)
    rows, V, k = 24, 30011, 200
    x = np.stack([group_row(rng, V, 2 + r % 6, r % 3, k) for r in range(rows)])
    hists = []
    for r in range(rows):
        top = np.argsort(-x[r], kind="stable")
        hists.append(np.concatenate([top[:1 + r % 3], top[20:60:2], rng.integers(0, V, 40)]).astype(np.int32))
        # (equal after the penalty too: the penalised members stay equal among themselves)
    ids = np.concatenate(hists)
    off = np.cumsum([0] + [h.size for h in hists]).astype(np.int64)
    pens = [dict(repetitionPenalty=1.01), dict(repetitionPenalty=1.02, presencePenalty=0.05,
                                               frequencyPenalty=0.01), dict(repetitionPenalty=0.9)]
    cfgs = [dict(dict(temperature=0.3, topK=k, topP=1.0), **pens[r % 3]) for r in range(rows)]
    u = rng.random(rows) * 0.9
    got = run_gpu(sampler, x, V, ids, off, cfgs, u, 64, want_cands=False)
    want, ref = run_oracle(x, V, ids, off, cfgs, u, 64)
    compare(got, want, ref, cfgs, V, 64, "equal values, penalised")
    assert (got.flags & 0x2).any()
    st = DecodeState(sampler, [h.tolist() for h in hists], (), ring_cap=256)
    d_l, d_u = hip.DeviceArray.from_numpy(x), hip.DeviceArray.from_numpy(u)
    d_t = hip.DeviceArray(rows, np.int32)
    st.step(d_l.addr, V, V, cfgs, d_u.addr, d_t.addr)
    hip.synchronize()
    assert d_t.download().tolist() == got.tokens.tolist()
    assert np.array_equal(d_l.download().view(np.uint32), ref.view(np.uint32))
    st.free()


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
