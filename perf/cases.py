"""Performance cases of the token-sampling path: what a serving program calls once per decode step.

Every case is one call (or the two calls of one step) through ``voidinfer_amd``'s
public entry points on device-resident inputs, as a decode loop holds them: the
LM head's logits, the lanes' parameters, their token histories or penalty
states.  A case is a dict of plain values:

========  =====================================================================
kind      entry point
========  =====================================================================
greedy    ``ops.greedy_rows_device``: argmax rows
sample    ``ops.sample_rows``: the batched sampler over token histories
state     ``ops.sample_rows_state`` recording the sampled tokens in the lanes'
          penalty states, and ``PenaltyState.update`` taking them out again
          (a speculated step that is rolled back; the pass leaves the state as
          it found it)
topk      ``ops.topk_rows``: the draft's exact top-k ids, values and log-probs
scores    ``ops.sampled_scores``: the coupled draw of a verified block's rows
          and the gap of the drafted tokens
verify    ``vi_verify_rows``: sampled verification of drafted tokens
chain     ``ops.selector_chain``: the draft's selector chain
========  =====================================================================

Logits are N(0, std) plus, where ``zipf`` is set, a Zipf(1.1) bias of at most 8
over a random order of the token ids.  Rows of 16-bit logits are contiguous, so
an odd vocabulary makes rows that start off a 16-byte boundary.
"""
from __future__ import annotations

import math

import numpy as np
import torch

import voidinfer_amd as vi
from voidinfer_amd import ops

_DT = {"bf16": torch.bfloat16, "f16": torch.float16, "f32": torch.float32}
_ABI = {"bf16": vi.BF16, "f16": vi.F16, "f32": vi.F32}
_SIZE = {"bf16": 2, "f16": 2, "f32": 4}
_DEV = "cuda:0"


def listed():
    return [
        # One lane's greedy token: the smallest call there is, launch latency only.
        dict(name="greedy-1-f32", kind="greedy", rows=1, vocab=151936, dtype="f32"),
        # A greedy batch over an odd vocabulary: every second row starts off a 16-byte boundary.
        dict(name="greedy-64-bf16-odd", kind="greedy", rows=64, vocab=65537, dtype="bf16"),
        # One interactive lane: T .7 / top_k 20 / top_p .8, repetition 1.05 over 256 tokens.
        dict(name="sample-1-f32", kind="sample", rows=1, vocab=151936, dtype="f32", std=2.0, zipf=True, mix="chat",
             history=256, ragged=False, skew=1.0, probs=False),
        # A small batch in which every request brings its own parameters (top_k off, 20 or 50, all penalties).
        dict(name="sample-8-bf16-mixed", kind="sample", rows=8, vocab=248320, dtype="bf16", std=2.0, zipf=True,
             mix="mixed", history=4096, ragged=False, skew=1.0, probs=False),
        # Filtered distributions wanted beside the tokens (an independent-rejection drafter's q), ragged
        # histories with the repeats that text has.
        dict(name="sample-24-bf16-probs", kind="sample", rows=24, vocab=151936, dtype="bf16", std=2.0, zipf=True,
             mix="full", history=2048, ragged=True, skew=3.0, probs=True),
        # The headline decode step: 128 lanes, near-flat logits, top_p .95, 32,768 tokens generated per lane.
        dict(name="state-128-bf16", kind="state", rows=128, vocab=248320, dtype="bf16", std=0.1, zipf=False,
             mix="full", history=32768, skew=1.0, slots=65536),
        # A large batch over fp32 logits with no penalties: the most bytes of all cases.
        dict(name="sample-128-f32-full", kind="sample", rows=128, vocab=248320, dtype="f32", std=2.0, zipf=True,
             mix="plain", history=0, ragged=False, skew=1.0, probs=False),
        # The draft's candidates: exact top-8 and log-probs of 128 fp16 rows.
        dict(name="topk-128-f16", kind="topk", rows=128, vocab=248320, dtype="f16", std=1.5, zipf=True, k=8),
        # A verified block of 16 rows scored against its drafted tokens, presence penalty on.
        dict(name="scores-16-f16", kind="scores", rows=16, vocab=248320, dtype="f16", std=2.0, zipf=True),
        # Verification of 8 lanes x 16 drafted tokens (and the bonus row) over top-20 lists.
        dict(name="verify-8x16-list", kind="verify", lanes=8, drafts=16, bonus=True, vocab=248320, dtype="bf16",
             draft_dtype="f16", std=2.0, zipf=True, top_k=20, top_p=0.8),
        # The same with top_k off: p and q are full-vocabulary distributions.
        dict(name="verify-8x16-full", kind="verify", lanes=8, drafts=16, bonus=True, vocab=248320, dtype="bf16",
             draft_dtype="f16", std=2.0, zipf=True, top_k=0, top_p=0.8),
        # The draft's selector chain for 8 lanes x 16 positions: a chain of dependent gathers.
        dict(name="chain-8x16", kind="chain", lanes=8, positions=16, vocab=248320),
    ]


def _spread(rng, low, high):
    """A whole number spread over the logarithm of [low, high]."""
    return max(low, min(high, int(round(math.exp(rng.uniform(math.log(low), math.log(high)))))))


def _vocab(rng):
    v = _spread(rng, 32000, 248320)
    return v | 1 if rng.random() < 0.3 else v // 64 * 64


def draw(rng):
    kind = rng.choice(["greedy", "sample", "sample", "probs", "state", "topk", "scores", "verify", "verify", "chain"])
    vocab, dtype = _vocab(rng), rng.choice(["bf16", "f16", "f32"])
    std = round(rng.choice([0.1, rng.uniform(1.0, 3.0)]), 3)
    shape = dict(vocab=vocab, dtype=dtype, std=std, zipf=std >= 1.0)
    if kind == "greedy":
        return dict(kind="greedy", rows=_spread(rng, 1, 128), vocab=vocab, dtype=dtype)
    if kind == "sample":
        mix = rng.choice(["chat", "mixed", "full", "plain"])
        return dict(kind="sample", rows=_spread(rng, 1, 128), mix=mix, probs=False, ragged=rng.random() < 0.5,
                    history=0 if mix == "plain" else _spread(rng, 64, 32768), skew=rng.choice([1.0, 3.0]), **shape)
    if kind == "probs":
        return dict(kind="sample", rows=_spread(rng, 1, 24), mix=rng.choice(["mixed", "full"]), probs=True,
                    ragged=True, history=_spread(rng, 64, 8192), skew=rng.choice([1.0, 3.0]),
                    **{**shape, "vocab": min(vocab, 151936)})
    if kind == "state":
        return dict(kind="state", rows=_spread(rng, 1, 128), mix=rng.choice(["chat", "mixed", "full"]),
                    history=_spread(rng, 64, 32768), skew=rng.choice([1.0, 3.0]), slots=65536, **shape)
    if kind == "topk":
        return dict(kind="topk", rows=_spread(rng, 1, 128), k=rng.choice([1, 8, 16, 20, 64]), **shape)
    if kind == "scores":
        return dict(kind="scores", rows=_spread(rng, 1, 16), **{**shape, "std": max(std, 1.0), "zipf": True})
    if kind == "verify":
        drafts = rng.choice([3, 7, 15, 16])
        top_k = rng.choice([0, 20, 50])
        if top_k == 0:   # full-vocabulary distributions need rows on a 16-byte boundary
            shape["vocab"] = vocab // 64 * 64
        return dict(kind="verify", lanes=_spread(rng, 1, 128 // drafts), drafts=drafts, bonus=rng.random() < 0.7,
                    draft_dtype=rng.choice([dtype, "f16"]), top_k=top_k, top_p=rng.choice([0.8, 0.95]),
                    **{**shape, "std": max(std, 1.0), "zipf": True})
    return dict(kind="chain", lanes=_spread(rng, 1, 64), positions=rng.choice([4, 8, 15, 16]), vocab=vocab)


# ---- inputs -----------------------------------------------------------------


def _gaussian_zipf(g, rows, vocab, std, zipf):
    x = torch.randn(rows, vocab, generator=g, device=_DEV) * std
    if zipf:
        rank = torch.randperm(vocab, generator=g, device=_DEV).float() + 1.0
        bias = 8.0 / rank ** 1.1
        for r in range(rows):   # another order of the ids for each row
            x[r] += torch.roll(bias, (r * 7919) % vocab)
    return x


def _tokens(g, n, vocab, skew):
    """Token ids, uniform (skew 1) or with the repeats of text (skew 3: half of them from an eighth of the ids)."""
    u = torch.rand(n, generator=g, device=_DEV, dtype=torch.float64)
    return (u ** skew * vocab).long().clamp_(max=vocab - 1).int()


def _params(rng, rows, mix):
    p = vi.params_array(rows, seed=rng.integers(1, 2 ** 62, rows), position=4096)
    if mix == "chat":       # one set of parameters for everybody
        p["temperature"], p["top_k"], p["top_p"], p["repetition_penalty"] = 0.7, 20, 0.8, 1.05
    elif mix == "plain":    # nucleus sampling only
        p["temperature"], p["top_p"] = 0.7, 0.95
    else:                   # every request brings its own
        p["temperature"] = rng.uniform(0.3, 1.2, rows)
        p["repetition_penalty"] = rng.uniform(1.0, 1.1, rows)
        p["presence_penalty"] = rng.uniform(0.0, 0.5, rows)
        p["frequency_penalty"] = rng.uniform(0.0, 0.5, rows)
        p["top_p"] = 0.95
        if mix == "mixed":
            p["top_k"] = rng.choice(np.array([0, 20, 50], dtype=np.int32), rows)
            p["top_p"] = rng.choice(np.array([0.8, 0.95, 1.0], dtype=np.float32), rows)
            p["min_p"] = rng.choice(np.array([0.0, 0.05], dtype=np.float32), rows)
    return p


def _draw_from(g, x, temperature, top_k, top_p):
    """One token per row from the row's top-k / top-p filtered distribution."""
    z, ids = torch.sort(x / temperature, dim=1, descending=True, stable=True)
    if top_k:
        z, ids = z[:, :top_k], ids[:, :top_k]
    w = torch.softmax(z.double(), dim=1)
    cum = torch.cumsum(w, dim=1)
    mass = torch.where(cum - w < top_p, w, torch.zeros_like(w)).cumsum(dim=1)
    u = torch.rand(x.shape[0], 1, generator=g, device=_DEV, dtype=torch.float64) * mass[:, -1:]
    at = torch.searchsorted(mass, u, right=True).clamp_(max=z.shape[1] - 1)
    return torch.gather(ids, 1, at).squeeze(1).int()


def prepare(case, seed):
    g = torch.Generator(device=_DEV)
    g.manual_seed(seed)
    rng = np.random.default_rng(seed)
    kind, vocab = case["kind"], case["vocab"]
    s = dict(case=case)
    if kind == "chain":
        lanes, positions = case["lanes"], case["positions"]
        s["anchors"] = torch.randint(0, vocab, (lanes,), generator=g, device=_DEV)
        s["candidates"] = torch.randint(0, vocab, (lanes, positions, 16), generator=g, device=_DEV)
        unary = torch.randn(lanes, positions, 16, generator=g, device=_DEV)
        s["unary"] = torch.sort(unary, dim=2, descending=True).values.contiguous()
        s["hidden"] = torch.randn(lanes, positions, 256, generator=g, device=_DEV).half()
        s["pred"] = (torch.randn(vocab, 256, generator=g, device=_DEV) * 0.25).half()
        s["succ"] = (torch.randn(vocab, 256, generator=g, device=_DEV) * 0.25).half()
        return s
    if kind == "verify":
        lanes, drafts = case["lanes"], case["drafts"]
        trows = drafts + int(case["bonus"])
        d = _gaussian_zipf(g, lanes * drafts, vocab, case["std"], case["zipf"])
        of = torch.tensor([l * drafts + min(j, drafts - 1) for l in range(lanes) for j in range(trows)], device=_DEV)
        t = d[of] + torch.randn(lanes * trows, vocab, generator=g, device=_DEV) * 0.5
        s["target"], s["draft"] = t.to(_DT[case["dtype"]]), d.to(_DT[case["draft_dtype"]])
        s["drafted"] = _draw_from(g, s["draft"].float(), 0.7, case["top_k"], case["top_p"])
        p = vi.params_array(lanes, temperature=0.7, top_k=case["top_k"], top_p=case["top_p"], position=5000,
                            seed=rng.integers(1, 2 ** 62, lanes))
        s["params"] = vi.to_device_bytes(p, _DEV)
        s["mode"] = vi.VERIFY_SAMPLED_TOPK if case["top_k"] else vi.VERIFY_SAMPLED
        s["accepted"] = torch.empty(lanes, dtype=torch.int32, device=_DEV)
        s["committed"] = torch.empty(lanes, drafts + 1, dtype=torch.int32, device=_DEV)
        s["count"] = torch.empty(lanes, dtype=torch.int32, device=_DEV)
        s["flags"] = torch.empty(lanes, dtype=torch.int32, device=_DEV)
        nb = vi.load().vi_verify_workspace_bytes(lanes, drafts, vocab)
        s["workspace"] = torch.zeros(nb, dtype=torch.uint8, device=_DEV)
        return s
    rows = case["rows"]
    x = _gaussian_zipf(g, rows, vocab, case.get("std", 2.0), case.get("zipf", True))
    s["logits"] = x.to(_DT[case["dtype"]])
    if kind == "greedy":
        s["out"] = torch.empty(rows * 16, dtype=torch.uint8, device=_DEV)
    elif kind == "scores":
        table = torch.full((vocab,), vi.ABSENT_OCCURRENCE, dtype=torch.int32, device=_DEV)
        vi.presence_record(table, 0, _tokens(g, 1024, vocab, 3.0).long())
        s["table"] = table
        s["next"] = _draw_from(g, s["logits"].float(), 0.9, 20, 1.0).long()
        s["seed"] = int(rng.integers(1, 2 ** 62))
    elif kind in ("sample", "state"):
        p = _params(rng, rows, case["mix"])
        s["host_params"], s["routes"] = p, vi.route_mask(p)
        s["params"] = vi.to_device_bytes(p, _DEV)
        n = case["history"]
        if n:
            lens = rng.integers(n // 4, n + 1, rows) if case.get("ragged") else np.full(rows, n)
            s["offsets"] = torch.from_numpy(np.concatenate([[0], np.cumsum(lens)]).astype(np.int64)).to(_DEV)
            s["histories"] = _tokens(g, int(lens.sum()), vocab, case["skew"])
        s["outputs"] = ops.SampleOutputs(
            torch.empty(rows, dtype=torch.int32, device=_DEV), None,
            torch.empty(rows, vocab, dtype=torch.float32, device=_DEV) if case.get("probs") else None,
            torch.empty(rows * vi.SAMPLE_STATS.itemsize, dtype=torch.uint8, device=_DEV))
        if kind == "state":
            s["state"] = vi.PenaltyState(rows, vocab, case["slots"], _DEV)
            s["state"].update(s["histories"], s["offsets"])
    return s


# ---- one pass ----------------------------------------------------------------


def _sampled(o):
    """The whole of a sampler call's outputs: the stats records as their whole and their floating fields."""
    stats = o.stats.view(-1, vi.SAMPLE_STATS.itemsize)
    floats = stats.view(torch.float64)
    got = dict(tokens=o.tokens, counts=stats.view(torch.int32)[:, :4], mass=floats[:, 2], uniform=floats[:, 3])
    if o.probs is not None:
        got["probs"] = o.probs
    return got


def run(s):
    case = s["case"]
    kind = case["kind"]
    if kind == "greedy":
        ops.greedy_rows_device(s["logits"], s["out"], serial=7)
        return s["out"]
    if kind == "sample":
        return _sampled(ops.sample_rows(s["logits"], s["params"], s.get("histories"), s.get("offsets"),
                                        case["history"], outputs=s["outputs"], routes=s["routes"]))
    if kind == "state":
        o = ops.sample_rows_state(s["logits"], s["params"], s["state"], record=True, outputs=s["outputs"],
                                  routes=s["routes"])
        s["state"].update(o.tokens, sign=-1)
        return _sampled(o)
    if kind == "topk":
        ids, values, logprobs = ops.topk_rows(s["logits"], case["k"], logprobs=True)
        return dict(ids=ids, values=values, logprobs=logprobs)
    if kind == "scores":
        chosen, gap = ops.sampled_scores(s["logits"], s["next"], 0.9, 20, 0.95, 0.02, s["seed"], first_key=1024,
                                         tolerance=0.25, presence_penalty=0.5, first_occurrence=s["table"])
        return dict(chosen=chosen, gap=gap)
    if kind == "chain":
        return ops.selector_chain(s["anchors"], s["candidates"], s["unary"], s["hidden"], s["pred"], s["succ"])
    t, d, ws, vocab = s["target"], s["draft"], s["workspace"], case["vocab"]
    status = vi.load().vi_verify_rows(
        s["mode"], t.data_ptr(), _ABI[case["dtype"]], vocab, t.shape[0] // case["lanes"], d.data_ptr(),
        _ABI[case["draft_dtype"]], vocab, case["lanes"], case["drafts"], vocab, s["drafted"].data_ptr(),
        s["params"].data_ptr(), None, 0, s["accepted"].data_ptr(), s["committed"].data_ptr(), s["count"].data_ptr(),
        s["flags"].data_ptr(), ws.data_ptr(), ws.numel(), torch.cuda.current_stream().cuda_stream)
    if status != 0:
        raise vi.VIError(status, "vi_verify_rows")
    return dict(accepted=s["accepted"], committed=s["committed"], count=s["count"], flags=s["flags"])


# ---- what a pass cannot do without -------------------------------------------


def work(case):
    """Bytes: the logits once, the penalty inputs once, the outputs once.  Operations: one comparison or one
    exponential's multiply-add per logit (no contraction anywhere)."""
    kind, vocab = case["kind"], case["vocab"]
    if kind == "chain":
        at = case["lanes"] * case["positions"]
        # per position: 16 candidates' and the anchor's 256 fp16 codebook entries, the hidden row, ids and scores
        return dict(bytes=at * (17 * 512 + 512 + 16 * 12 + 8), flops=at * 16 * 256 * 3)
    if kind == "verify":
        target = case["lanes"] * (case["drafts"] + int(case["bonus"])) * vocab
        draft = case["lanes"] * case["drafts"] * vocab
        return dict(bytes=target * _SIZE[case["dtype"]] + draft * _SIZE[case["draft_dtype"]]
                    + case["lanes"] * (48 + case["drafts"] * 8 + 16), flops=2 * (target + draft))
    rows = case["rows"]
    n = rows * vocab
    logits = n * _SIZE[case["dtype"]]
    if kind == "greedy":
        return dict(bytes=logits + rows * 16, flops=n)
    if kind == "topk":
        return dict(bytes=logits + rows * case["k"] * 16, flops=2 * n)
    if kind == "scores":   # the first-occurrence table serves every row
        return dict(bytes=logits + vocab * 4 + rows * 20, flops=n)
    out = rows * (48 + 4 + 32) + (n * 4 if case.get("probs") else 0)
    if kind == "state":    # a presence bit per token and 8 bytes per repeated token (about an eighth of them)
        return dict(bytes=logits + n // 8 + rows * case["history"], flops=2 * n)
    share = 0.625 if case["ragged"] else 1.0
    return dict(bytes=int(logits + rows * case["history"] * 4 * share + out), flops=2 * n)


def tolerance(case):
    kind = case["kind"]
    if kind in ("greedy", "verify"):
        return "exact"
    if kind == "chain":    # fp32 sums of 256 products: two candidates within their rounding may change places
        return dict(rel=0.0, differ=0.005)
    if kind == "topk":     # fp32 log-sum-exp of the row
        return dict(rel=2e-6, max=1e-5, differ=0.0)
    if kind == "scores":   # fp32 perturbed values (up to about 40) subtracted from one another
        return dict(rel=1e-5, max=1e-4, differ=0.0)
    # Masses: fp32 weights summed in fixed point or 64 bits.  A cut or a draw within the sums' rounding of a
    # boundary may move by one token; counts hold the support, which is hundreds of thousands on flat rows.
    return dict(rel=2e-6, max=2e-5, differ=0.01 if case["rows"] >= 24 else 0.0)


# ---- the same in 64 bits -----------------------------------------------------


def _penalized(case, s):
    """z = penalized logit / T per row, in the 32-bit steps that the sampler is defined by."""
    x = s["logits"].float()
    p = s["host_params"]
    col = lambda k: torch.from_numpy(p[k].copy()).to(_DEV)[:, None]   # noqa: E731
    if case["history"]:
        offs, h = s["offsets"].tolist(), s["histories"].long()
        count = torch.stack([torch.bincount(h[a:b], minlength=case["vocab"]) for a, b in zip(offs, offs[1:])])
        rep = col("repetition_penalty")
        y = torch.where(x > 0, x / rep, x * rep)
        y = y - col("frequency_penalty") * count.float()
        y = (y - col("presence_penalty")).to(s["logits"].dtype).float()
        x = torch.where(count > 0, y, x)
    return x * (1.0 / col("temperature"))


def _gumbel(seed, key, token):
    m = (1 << 64) - 1

    def mix(v):
        v = (v + 0x9E3779B97F4A7C15) & m
        v = ((v ^ (v >> 30)) * 0xBF58476D1CE4E5B9) & m
        v = ((v ^ (v >> 27)) * 0x94D049BB133111EB) & m
        return v ^ (v >> 31)
    h = mix(seed ^ (key * 0xD1B54A32D192ED03 & m))
    h = mix(h ^ (token * 0x2545F4914F6CDD1D & m))
    return -math.log(-math.log(((h >> 40) + 0.5) / 16777216.0))


def _support(w, min_p, top_p):
    cum, total = 0.0, sum(w)
    for j, v in enumerate(w):
        if min_p > 0 and v < min_p * w[0]:
            return max(1, j)
        cum += v
        if top_p < 1 and cum >= top_p * total:
            return j + 1
    return len(w)


def _exact_gap(s, row, vocab):
    temp, top_p, min_p = (float(np.float32(v)) for v in (0.9, 0.95, 0.02))
    inv = float(np.float32(1.0) / np.float32(0.9))
    key = 1024 + row
    x = s["logits"][row].float() - 0.5 * (s["table"] < key)
    val, idx = torch.sort(x, descending=True, stable=True)
    val, idx = val[:20].double().tolist(), idx[:20].tolist()
    want = int(s["next"][row])
    weigh = lambda v: [math.exp((a - v[0]) * inv) for a in v]   # noqa: E731
    n = _support(weigh(val), min_p, top_p)
    value = [v * inv + _gumbel(s["seed"], key, i) for v, i in zip(val, idx)]
    best = max(range(n), key=lambda j: value[j])
    if idx[best] == want:
        return 0.0
    if want not in idx:
        return math.inf
    rank = idx.index(want)
    if rank < n:
        return (value[best] - value[rank]) * temp
    raised = val[rank] + 0.25
    rest = [(v, i) for j, (v, i) in enumerate(zip(val, idx)) if j != rank]
    at = sum(1 for v, _ in rest if v >= raised)
    rest.insert(at, (raised, want))
    n = _support(weigh([v for v, _ in rest]), min_p, top_p)
    if at >= n:
        return math.inf
    others = max((v * inv + _gumbel(s["seed"], key, i) for j, (v, i) in enumerate(rest[:n]) if j != at),
                 default=-math.inf)
    return max(0.0, (others - value[rank]) * temp)


def exact(case, seed):
    kind, vocab = case["kind"], case["vocab"]
    if kind in ("greedy", "verify", "chain"):
        return None   # tokens and counts only
    s = prepare(case, seed)
    if kind == "topk":
        x = s["logits"].double()
        values = torch.sort(x, dim=1, descending=True).values[:, :case["k"]]
        return dict(ids=None, values=values, logprobs=values - torch.logsumexp(x, dim=1, keepdim=True))
    if kind == "scores":
        gap = [_exact_gap(s, r, vocab) for r in range(case["rows"])]
        return dict(chosen=None, gap=torch.tensor(gap, dtype=torch.float64))
    z, ids = torch.sort(_penalized(case, s), dim=1, descending=True, stable=True)
    mass, probs = [], []
    for r, p in enumerate(s["host_params"]):
        k = int(p["top_k"]) or vocab
        w = torch.exp(z[r, :k].double() - z[r, 0].double())
        cum = torch.cumsum(w, 0)
        n = k
        if p["min_p"] > 0:
            n = min(n, int((w >= float(p["min_p"])).sum()))
        if p["top_p"] < 1:
            n = min(n, int((cum < float(p["top_p"]) * cum[-1]).sum()) + 1)
        n = max(1, n)
        mass.append(w[:n].sum())
        if case.get("probs"):
            row = torch.zeros(vocab, dtype=torch.float64, device=_DEV)
            row[ids[r, :n]] = w[:n] / mass[-1]
            probs.append(row)
    got = dict(tokens=None, counts=None, mass=torch.stack(mass), uniform=None)
    if probs:
        got["probs"] = torch.stack(probs)
    return got
