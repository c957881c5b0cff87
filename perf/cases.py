"""Performance cases of the gfx950 sampler and its lm_head, through the
Python entry points (hachiue_amd.Sampler) on device-resident buffers, the way
a decode loop calls them once per step.

Five kinds of pass:
  sample   Sampler.sample_device: penalties, top-k / top-p / min-p and the draw
           over rows of float32 logits, each with its token history
  argmax   Sampler.argmax_device: the engine's greedy route
  lm_head  Sampler.gemv_device_ex: logits of M hidden states from a weight
           tensor in one of the GGUF formats
  lm_head_sample  Sampler.lm_head_sample_device_ex: both, in one call
  decode   gemv_device_ex, then Sampler.decode_step_device: the next step of M
           running sequences with their histories in device rings

One Sampler serves the whole process, as a server keeps one.  Options are a
function of the case alone (a batch keeps its options from step to step);
logits, weights, hidden states, histories and uniforms come from the seed.
"""
import numpy as np
import torch

from hachiue_amd import Sampler
from hachiue_amd.sampler import make_configs, weights

INF = float("inf")
V = 151936                    # the workloads' vocabulary (262144 is the other)
RING = 4096                   # ids a decode ring keeps

# format: (GGML type, weights per block, bytes per block as held on the GPU)
FORMATS = {"f32": (0, 1, 4), "q4_0": (2, 32, 18), "q4_1": (3, 32, 20), "q4_k": (12, 256, 144),
           "q6_k": (14, 256, 210), "q1_0": (41, 128, 18), "pq2_0": (142, 128, 34),
           "ptq1_0": (143, 128, 28)}
PLANAR = {"q1_0": 16, "pq2_0": 32, "ptq1_0": 26}     # quant bytes per block

# what a drawn case may cost at most, from the largest listed ones: logits,
# weight bytes, weight bytes and weights times hidden states
MAX_LOGITS = 1024 * V
MAX_WEIGHTS = 640 << 20
MAX_WORK = 48 * (V * 2048 // 256 * 210)
MAX_PRODUCTS = 40 * V * 2048


def listed():
    return [
        # one sequence, the reference's own use: one row per decode step
        # (top-k 40, top-p 0.9, repetition 1.1 over 64 ids); the smallest call
        dict(name="sample-1", kind="sample", rows=1, vocab=V, style="topk", hist=64),
        # a small serving batch, longer histories
        dict(name="sample-64", kind="sample", rows=64, vocab=V, style="topk", hist=256),
        # the benchmark's default batch
        dict(name="sample-256", kind="sample", rows=256, vocab=V, style="topk", hist=64),
        # every row with options of its own: top-k up to 1024, top-p,
        # temperature, presence and frequency over the whole history
        dict(name="perrow-256", kind="sample", rows=256, vocab=V, style="perrow", hist=1024),
        # a large batch on the larger vocabulary, all penalties, top-k 100
        dict(name="penalties-512", kind="sample", rows=512, vocab=262144, style="pen", hist=4096),
        # nucleus sampling without top-k over flat (Gumbel) logits
        dict(name="topp-1024", kind="sample", rows=1024, vocab=V, style="topp", hist=0),
        # min-p sampling without top-k on a ragged batch
        dict(name="minp-50", kind="sample", rows=50, vocab=V, style="minp", hist=200),
        # one sequence's lm_head in the formats its models ship in
        dict(name="lm-head-q6k-1", kind="lm_head", fmt="q6_k", m=1, vocab=V, hidden=2048,
             hadamard=False),
        dict(name="lm-head-q4_0-1", kind="lm_head", fmt="q4_0", m=1, vocab=V, hidden=1024,
             hadamard=False),
        # a ternary lm_head with the Hadamard fold and greedy decoding: one sequence
        dict(name="greedy-ptq1-1", kind="lm_head_sample", fmt="ptq1_0", m=1, vocab=V, hidden=2048,
             hadamard=True, style="greedy", hist=64),
        # a few sequences decoded together
        dict(name="lm-head-sample-q4k-7", kind="lm_head_sample", fmt="q4_k", m=7, vocab=V,
             hidden=4096, hadamard=False, style="topk", hist=300),
        # a batch's whole step: lm_head, draw, stop check, history append
        dict(name="decode-q6k-64", kind="decode", fmt="q6_k", m=64, vocab=V, hidden=2048,
             hadamard=False, style="topk", hist=200),
    ]


def _log(rng, lo, hi):
    return int(round(lo * (hi / lo) ** rng.random()))


def draw(rng):
    kind = rng.choice(["sample", "sample", "argmax", "lm_head", "lm_head_sample", "decode"])
    vocab = V if rng.random() < 0.3 else _log(rng, 32000, 262144)
    if kind in ("sample", "argmax"):
        rows = min(_log(rng, 1, 1024), MAX_LOGITS // vocab)
        if kind == "argmax":
            return dict(kind=kind, rows=rows, vocab=vocab)
        style = rng.choice(["topk", "topk", "perrow", "pen", "topp", "minp", "greedy"])
        return dict(kind=kind, rows=rows, vocab=vocab, style=style, hist=_log(rng, 1, 4096))
    fmt = rng.choice(sorted(FORMATS))
    hidden = 512 * rng.randint(1, 8)
    _, bw, bb = FORMATS[fmt]
    vocab = min(vocab, MAX_WEIGHTS // (hidden // bw * bb))
    m = min(_log(rng, 1, 64), max(1, MAX_WORK // (vocab * (hidden // bw) * bb)),
            MAX_PRODUCTS // (vocab * hidden))
    c = dict(kind=kind, fmt=fmt, m=m, vocab=vocab, hidden=hidden, hadamard=rng.random() < 0.3)
    if kind != "lm_head":
        c.update(style=rng.choice(["topk", "topk", "perrow", "greedy"]), hist=_log(rng, 1, 2048))
    return c


# ---- inputs ---------------------------------------------------------------

_SAMPLER = None


def _sampler():
    global _SAMPLER
    if _SAMPLER is None:
        _SAMPLER = Sampler(0)
    return _SAMPLER


def _options(style, rows):
    """The batch's SampleConfigs."""
    if style == "greedy":
        return [dict(temperature=0.0, repetitionPenalty=1.1)] * rows
    if style == "topk":
        return [dict(temperature=0.7, topK=40, topP=0.9, repetitionPenalty=1.1)] * rows
    if style == "pen":
        return [dict(temperature=0.9, topK=100, topP=0.9, repetitionPenalty=1.15,
                     presencePenalty=0.4, frequencyPenalty=0.2)] * rows
    if style == "topp":
        return [dict(temperature=1.0, topK=INF, topP=0.98)] * rows
    if style == "minp":
        return [dict(temperature=1.0, topK=INF, topP=1.0, minP=0.05, repetitionPenalty=1.1)] * rows
    r = np.random.default_rng(rows)     # perrow
    return [dict(temperature=float(r.uniform(0.3, 1.5)), topK=int(r.integers(1, 1025)),
                 topP=float(r.uniform(0.5, 0.99)), presencePenalty=0.5, frequencyPenalty=0.3)
            for _ in range(rows)]


def _generator(case, seed):
    g = torch.Generator("cuda")
    g.manual_seed(seed * 7919 + case["vocab"])
    return g


def _logits(case, g):
    rows, vocab = case["rows"], case["vocab"]
    if case.get("style") == "topp":     # standard Gumbel
        x = torch.empty(rows, vocab, device="cuda").exponential_(generator=g)
        return x.clamp_(min=1e-30).log_().neg_()
    x = torch.empty(rows, vocab, device="cuda").normal_(0.0, 2.5, generator=g)
    # a model's few likely tokens
    top = torch.randint(0, vocab, (rows, 8), device="cuda", generator=g)
    return x.scatter_add_(1, top, torch.full((rows, 8), 12.0, device="cuda"))


def _histories(rows, n, vocab, g):
    """[rows, n] ids with the repeats of text: Zipf(1.1) ranks over a shuffled
    vocabulary."""
    p = torch.arange(1, vocab + 1, device="cuda", dtype=torch.float64) ** -1.1
    cdf = torch.cumsum(p, 0)
    u = torch.rand(rows, n, device="cuda", dtype=torch.float64, generator=g) * cdf[-1]
    rank = torch.searchsorted(cdf, u).clamp_(max=vocab - 1)
    return torch.randperm(vocab, device="cuda", generator=g)[rank].to(torch.int32)


def _binary16(shape, scale, g):
    """Positive binary16 block scales around `scale`, as bytes [..., 2]."""
    d = (torch.rand(shape, device="cuda", generator=g) + 0.5) * scale
    return d.to(torch.float16).unsqueeze(-1).view(torch.uint8)


def _weight_bytes(case, g):
    """(quants or whole blocks [vocab, blocks, bytes], planar binary16 scales
    or None).  Random quants; scales that give logits a standard deviation of
    about 2.5, as the sampling cases have."""
    fmt, vocab, K = case["fmt"], case["vocab"], case["hidden"]
    _, bw, bb = FORMATS[fmt]
    nb = K // bw
    rms = 1.8 / K ** 0.5           # of a weight (hidden states have rms 1.4)
    if fmt == "f32":
        w = torch.empty(vocab, K, device="cuda").normal_(0.0, rms, generator=g)
        return w, None
    if fmt in PLANAR:
        q = torch.randint(0, 256, (vocab, nb, PLANAR[fmt]), device="cuda", dtype=torch.uint8,
                          generator=g)
        return q, _binary16((vocab, nb), rms, g)
    q = torch.randint(0, 256, (vocab, nb, bb), device="cuda", dtype=torch.uint8, generator=g)
    if fmt == "q4_0":
        q[:, :, 0:2] = _binary16((vocab, nb), rms / 4.6, g)
    elif fmt == "q4_1":
        q[:, :, 0:2] = _binary16((vocab, nb), rms / 4.6, g)
        q[:, :, 2:4] = _binary16((vocab, nb), rms / 4.6 * 7.5, g)
        q[:, :, 3] |= 0x80         # minima lie below zero
    elif fmt == "q4_k":
        q[:, :, 0:2] = _binary16((vocab, nb), rms / 200.0, g)
        q[:, :, 2:4] = _binary16((vocab, nb), rms / 200.0 * 7.5, g)
    else:
        q[:, :, 208:210] = _binary16((vocab, nb), rms / 1369.0, g)
    return q, None


def _hidden_states(case, g):
    """A final norm's output: unit normal with one channel in a hundred ten
    times as large."""
    m, K = case["m"], case["hidden"]
    big = torch.rand(K, device="cuda", generator=g) < 0.01
    x = torch.empty(m, K, device="cuda").normal_(0.0, 1.0, generator=g)
    return torch.where(big, x * 10.0, x).contiguous()


def _inputs(case, seed):
    g = _generator(case, seed)
    s = dict(case=dict(case))
    if case["kind"] in ("sample", "argmax"):
        rows = case["rows"]
        s["logits"] = _logits(case, g)
    else:
        rows = case["m"]
        s["x"] = _hidden_states(case, g)
        s["w"], s["scales"] = _weight_bytes(case, g)
        s["signs"] = (torch.randint(0, 2, (case["hidden"],), device="cuda", generator=g)
                      .float().mul_(2.0).sub_(1.0)) if case["hadamard"] else None
        s["logits"] = torch.empty(rows, case["vocab"], device="cuda")
    s["rows"] = rows
    if "style" in case:
        s["hist"] = _histories(rows, case["hist"], case["vocab"], g) if case["hist"] else None
        s["u"] = torch.rand(rows, device="cuda", dtype=torch.float64, generator=g)
    return s


def prepare(case, seed):
    s = _inputs(case, seed)
    rows = s["rows"]
    s["sampler"] = _sampler()
    s["stream"] = torch.cuda.current_stream().cuda_stream
    s["tokens"] = torch.zeros(rows, dtype=torch.int32, device="cuda")
    if "style" in case:
        s["configs"] = make_configs(_options(case["style"], rows), rows)
    if case["kind"] == "decode":
        n = case["hist"]
        s["ring"] = torch.zeros(rows, RING, dtype=torch.int32, device="cuda")
        s["ring"][:, :n] = s["hist"]
        s["len"] = torch.full((rows,), n, dtype=torch.int64, device="cuda")
        s["done"] = torch.zeros(rows, dtype=torch.int32, device="cuda")
        s["stop"] = torch.tensor([case["vocab"] - 1, case["vocab"] - 2], dtype=torch.int32,
                                 device="cuda")
    elif s.get("hist") is not None:
        s["off"] = torch.arange(rows + 1, dtype=torch.int64, device="cuda") * case["hist"]
    if "w" in s:
        s["weights"] = weights(FORMATS[case["fmt"]][0], case["vocab"], case["hidden"],
                               s["w"].data_ptr(),
                               s["scales"].data_ptr() if s["scales"] is not None else None,
                               case["hadamard"],
                               s["signs"].data_ptr() if s["signs"] is not None else None)
    return s


def run(s):
    c, smp, st = s["case"], s["sampler"], s["stream"]
    vocab, rows = c["vocab"], s["rows"]
    logits, tokens = s["logits"], s["tokens"]
    ids = s["hist"].data_ptr() if s.get("hist") is not None else None
    off = s["off"].data_ptr() if "off" in s else None
    if c["kind"] == "sample":
        smp.sample_device(logits.data_ptr(), rows, vocab, vocab, ids, off, s["configs"],
                          s["u"].data_ptr(), tokens.data_ptr(), stream=st)
    elif c["kind"] == "argmax":
        smp.argmax_device(logits.data_ptr(), rows, vocab, vocab, tokens.data_ptr(), stream=st)
        return tokens
    elif c["kind"] == "lm_head":
        smp.gemv_device_ex(s["x"].data_ptr(), rows, c["hidden"], s["weights"], logits.data_ptr(),
                           vocab, stream=st)
        return logits
    elif c["kind"] == "lm_head_sample":
        smp.lm_head_sample_device_ex(s["x"].data_ptr(), rows, c["hidden"], s["weights"],
                                     logits.data_ptr(), vocab, ids, off, s["configs"],
                                     s["u"].data_ptr(), tokens.data_ptr(), stream=st)
    else:
        smp.gemv_device_ex(s["x"].data_ptr(), rows, c["hidden"], s["weights"], logits.data_ptr(),
                           vocab, stream=st)
        smp.decode_step_device(logits.data_ptr(), rows, vocab, vocab, s["ring"].data_ptr(), RING,
                               s["len"].data_ptr(), s["done"].data_ptr(), s["stop"].data_ptr(), 2,
                               s["configs"], s["u"].data_ptr(), tokens.data_ptr(), stream=st)
        return dict(logits=logits, tokens=tokens, ring=s["ring"], len=s["len"], done=s["done"])
    return dict(logits=logits, tokens=tokens)


# ---- what a pass cannot do without ------------------------------------------

def work(case):
    """Logits (or weights and hidden states) and histories read once; logits
    of an lm_head, the penalised entries and the tokens written once."""
    rows, vocab = case.get("rows", case.get("m")), case["vocab"]
    n = rows * 4
    flops = 0
    if "fmt" in case:
        _, bw, bb = FORMATS[case["fmt"]]
        n += vocab * (case["hidden"] // bw) * bb + 4 * rows * case["hidden"] + 4 * rows * vocab
        flops = 2 * rows * vocab * case["hidden"]
    else:
        n += 4 * rows * vocab
    if "style" in case:
        n += rows * 4 * (case["hist"] if case["style"] in ("perrow", "pen") else
                         0 if case["style"] == "topp" else min(case["hist"], 128))
    return dict(bytes=n, flops=flops)


def tolerance(case):
    # penalised logits are defined bit for bit, and so are the ids; the rows
    # without a top-k sum their probabilities in an order of their own: a draw
    # that close to a boundary may give the neighbouring id (2 of 1024 rows)
    if "fmt" not in case:
        return {"rel": 0.0, "differ": 0.004} if case.get("style") in ("topp", "minp") else "exact"
    # lm_heads: binary32 sums of up to 4096 products
    return {"rel": 1e-6, "differ": 0.0}


# ---- the same in 64 bits ------------------------------------------------------

def _half(b):
    return b.contiguous().view(torch.float16).double()


def _trits(b, count):
    """The first `count` base-3 digits of each byte, digit by digit."""
    out = []
    for n in range(count):
        out.append((((b.int() * 3 ** n) & 0xFF) * 3) >> 8)
    return torch.cat(out, -1).double()


def _dequantised(fmt, w, scales):
    """[rows, hidden] binary64 weights of a slab of rows."""
    if fmt == "f32":
        return w.double()
    n, nb = w.shape[0], w.shape[1]
    if fmt in PLANAR:
        d = _half(scales)
        if fmt == "q1_0":
            bits = torch.arange(8, device="cuda")
            c = ((w.unsqueeze(-1).int() >> bits) & 1).reshape(n, nb, 128).double() * 2 - 1
        elif fmt == "pq2_0":
            sh = torch.arange(0, 8, 2, device="cuda")
            c = ((w.unsqueeze(-1).int() >> sh) & 3).reshape(n, nb, 128).double() - 1
        else:
            c = torch.cat([_trits(w[..., :16], 5), _trits(w[..., 16:24], 5),
                           _trits(w[..., 24:26], 4)], -1) - 1
        return (c * d).reshape(n, -1)
    d = _half(w[..., 208:210]) if fmt == "q6_k" else _half(w[..., 0:2])
    if fmt in ("q4_0", "q4_1"):
        b = w[..., 2:] if fmt == "q4_0" else w[..., 4:]
        q = torch.cat([b & 15, b >> 4], -1).double()
        q = (q - 8) * d if fmt == "q4_0" else q * d + _half(w[..., 2:4])
        return q.reshape(n, -1)
    if fmt == "q4_k":
        s = w[..., 4:16].int()
        sc = torch.cat([s[..., 0:4] & 63, (s[..., 8:12] & 15) | (s[..., 0:4] >> 6 << 4)], -1)
        mn = torch.cat([s[..., 4:8] & 63, (s[..., 8:12] >> 4) | (s[..., 4:8] >> 6 << 4)], -1)
        b = w[..., 16:].reshape(n, nb, 4, 1, 32)
        q = torch.cat([b & 15, b >> 4], 3).reshape(n, nb, 8, 32).double()
        v = (d * sc).unsqueeze(-1) * q - (_half(w[..., 2:4]) * mn).unsqueeze(-1)
        return v.reshape(n, -1)
    ql = w[..., :128].reshape(n, nb, 2, 2, 32)          # half, quarter & 1, position
    ql = torch.stack([ql & 15, ql >> 4], 3)             # half, quarter >> 1, quarter & 1, position
    ql = ql.reshape(n, nb, 2, 4, 32).int()
    sh = torch.arange(0, 8, 2, device="cuda").view(4, 1)
    qh = (w[..., 128:192].reshape(n, nb, 2, 1, 32).int() >> sh) & 3
    q = (ql | (qh << 4)).double() - 32
    sc = w[..., 192:208].contiguous().view(torch.int8).double().reshape(n, nb, 16, 1)
    return (q.reshape(n, nb, 16, 16) * sc * d.unsqueeze(-1)).reshape(n, -1)


def _hadamard(x, signs):
    m, K = x.shape
    x = (x * signs.double()).reshape(m, K // 512, 512)
    h = 1
    while h < 512:
        x = x.reshape(m, K // 512, 512 // (2 * h), 2, h)
        x = torch.stack([x[..., 0, :] + x[..., 1, :], x[..., 0, :] - x[..., 1, :]], 3)
        h *= 2
    return x.reshape(m, K) / 512 ** 0.5


def _penalised(y, hist, o):
    """One row's penalties: repetition over the last 128 ids, presence and
    frequency over all of them."""
    ids, n = torch.unique(hist, return_counts=True)
    v = y[ids.long()]
    rep = o.get("repetitionPenalty", 1.0)
    if rep != 1.0:
        last = torch.isin(ids, hist[-128:])
        v = torch.where(last, torch.where(v < 0, v * rep, v / rep), v)
    v = v - o.get("frequencyPenalty", 0.0) * n - o.get("presencePenalty", 0.0)
    y[ids.long()] = v


def exact(case, seed):
    """What run() returns first on these inputs, logits in binary64."""
    if case["kind"] == "argmax":
        return None
    s = _inputs(case, seed)
    if "fmt" in case:
        x = s["x"].double()
        if case["hadamard"]:
            x = _hadamard(x, s["signs"])
        y = torch.empty(s["rows"], case["vocab"], dtype=torch.float64, device="cuda")
        for a in range(0, case["vocab"], 16384):
            sc = s["scales"][a:a + 16384] if s["scales"] is not None else None
            w = _dequantised(case["fmt"], s["w"][a:a + 16384], sc)
            y[:, a:a + 16384] = x @ w.t()
    else:
        y = s["logits"].double()
    if case["kind"] == "lm_head":
        return y
    if s["hist"] is not None:
        for r, o in enumerate(_options(case["style"], s["rows"])):
            _penalised(y[r], s["hist"][r], o)
    out = dict(logits=y, tokens=None)
    if case["kind"] == "decode":
        out.update(ring=None, len=None, done=None)
    return out
