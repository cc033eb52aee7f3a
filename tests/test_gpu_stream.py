"""GPU full-vocabulary rows in one launch (csrc/sample_stream.hip) vs the CPU oracle.

The stream route serves the 16-bit full-route rows (temperature > 0, top_k 0 or
> 64) of vi_sample_rows / vi_sample_rows_state.  Bar: token ids equal to the
oracle's except where a cumulative-mass boundary lies within 1e-6 of the drawn
uniform or of a cut; support sizes, finite counts and flags equal
outside exempt rows; Philox uniforms bit-exact; support mass within 1e-6.
Cases: vocabularies from 64 to 248,320 and part boundaries (parts of up to 65,504 tokens),
one to 128 rows (one to sixteen parts per row), caps above 64, min-p, top-p,
ties, non-finite and empty rows, signed zeros, logits outside the fast
division's range, temperatures whose z overflows, repetition / presence /
frequency penalties from histories (the history view) and from penalty states
over recorded decode steps, tokens seen hundreds of times, bad history tokens,
and repeated calls on one workspace (the self-resetting counters).
"""
import numpy as np
import pytest
import torch

from helpers import exempt_draw, to_dev
from test_gpu_sample import compare, make_rows, params, run_both

pytestmark = pytest.mark.gpu


def stream(orc, dev, bits, dtype, p, hist=None, offs=None, label=""):
    print(f"[stream] {label} rows={len(p)} vocab={bits.shape[1]}", flush=True)
    return compare(*run_both(orc, dev, bits, dtype, p, hist, offs, want_probs=False), p, label)


@pytest.mark.parametrize("dtype", [0, 1])
@pytest.mark.parametrize("vocab", [64, 1024, 65_528, 65_536, 131_072, 248_320])
def test_stream_filters(orc, dev, rng, dtype, vocab):
    rows = 16
    bits = make_rows(rng, rows, vocab, std=1.0, dtype=dtype)
    p = params(rows, rng, temperature=rng.uniform(0.3, 1.2, rows), top_k=rng.choice([0, 0, 100, 1000], rows),
               top_p=rng.choice([0.5, 0.9, 0.95, 1.0], rows), min_p=rng.choice([0.0, 0.0, 0.01, 0.1], rows))
    stream(orc, dev, bits, dtype, p, label=f"filters-{dtype}-{vocab}")


@pytest.mark.parametrize("rows", [1, 2, 3, 8, 9])
def test_stream_small_batches(orc, dev, rng, rows):
    """Few rows: up to sixteen parts per row, parts spread over every XCD."""
    vocab = 248_320
    bits = make_rows(rng, rows, vocab, std=2.0)
    p = params(rows, rng, temperature=rng.uniform(0.5, 1.0, rows), top_k=0, top_p=rng.choice([0.8, 0.95], rows))
    stream(orc, dev, bits, 0, p, label=f"small-{rows}")


@pytest.mark.parametrize("dtype", [0, 1])
def test_stream_penalties_and_saturation(orc, dev, rng, dtype):
    rows, vocab = 8, 100_000
    bits = make_rows(rng, rows, vocab, std=0.5, dtype=dtype)
    p = params(rows, rng, temperature=rng.uniform(0.5, 1.2, rows), top_k=0, top_p=rng.choice([0.9, 0.95], rows),
               repetition_penalty=rng.uniform(1.0, 1.2, rows), presence_penalty=rng.uniform(0, 0.5, rows),
               frequency_penalty=rng.uniform(0, 0.05, rows))
    L = 6000
    rows_h = []
    for r in range(rows):
        h = rng.integers(0, vocab, L).astype(np.int32)
        h[:600] = 77                     # one token seen 600 times
        h[600:900] = vocab - 1           # ... and one at the last id of the row
        h[900:1000] = rng.integers(0, 50, 100)
        rows_h.append(h)
    offs = np.arange(rows + 1, dtype=np.int64) * L
    stream(orc, dev, bits, dtype, p, np.concatenate(rows_h), offs, "penalties")


@pytest.mark.parametrize("dtype", [0, 1])
def test_stream_repeated_history_tokens(orc, dev, rng, dtype):
    """Tokens seen 2..7 times and at part boundaries: the count-1 penalty of the
    stream corrected from the repeat list at the end of each part."""
    rows, vocab = 8, 248_320
    bits = make_rows(rng, rows, vocab, std=0.5, dtype=dtype)
    p = params(rows, rng, temperature=rng.uniform(0.5, 1.2, rows), top_k=0, top_p=rng.choice([0.9, 0.95], rows),
               repetition_penalty=rng.uniform(1.0, 1.3, rows), presence_penalty=rng.uniform(0, 0.5, rows),
               frequency_penalty=rng.uniform(0.05, 0.3, rows))
    rows_h = []
    for r in range(rows):
        pool = rng.choice(vocab, 400, replace=False)
        reps = np.concatenate([np.repeat(pool[:300], 2 + r % 3), np.repeat(pool[300:], 7)])
        edges = [15_519, 15_520, 62_079, 62_080, 124_159, 124_160, vocab - 1]
        h = np.concatenate([rng.integers(0, vocab, 3000), reps, np.repeat(edges, 3)])
        rows_h.append(rng.permutation(h).astype(np.int32))
    offs = np.concatenate([[0], np.cumsum([len(h) for h in rows_h])]).astype(np.int64)
    stream(orc, dev, bits, dtype, p, np.concatenate(rows_h), offs, "repeats")


def test_stream_nonfinite_and_ties(orc, dev, rng):
    rows, vocab = 6, 9_000
    bits = make_rows(rng, rows, vocab, std=1.0)
    bits[0, ::7] = 0x7FC0          # NaN
    bits[1, 5] = 0x7F80            # +inf
    bits[2, :] = 0x3F80            # all equal (1.0): pure tie-break by id
    bits[3, :4000] = 0x3F80
    bits[4, :] = 0x7FC0            # nothing finite
    p = params(rows, rng, temperature=0.9, top_k=0, top_p=rng.choice([0.3, 0.9], rows))
    g, w = run_both(orc, dev, bits, 0, p, want_probs=False)
    compare(g, w, p, "nonfinite")
    assert w["stats"]["flags"][4] & 2 and g["tokens"][4] == vocab


def test_stream_signed_zeros_extremes_and_temperatures(orc, dev, rng):
    """+0 / -0 (one key), logits beyond the fast division's range (|x| > 2^100,
    subnormal), temperatures whose z overflows, and T > 65,536 (refused)."""
    rows, vocab = 8, 4_096
    bits = make_rows(rng, rows, vocab, std=1.0)
    bits[0, ::2] = 0x0000
    bits[0, 1::2] = 0x8000
    bits[1, :64] = 0x7F00                          # 1.7e38
    bits[1, 64:128] = 0x0001                       # subnormal
    bits[2, :200] = 0x7F00
    bits[3, ::3] = 0x8000
    hist = np.concatenate([np.arange(0, 256, dtype=np.int32)] * rows)
    offs = np.arange(rows + 1, dtype=np.int64) * 256
    p = params(rows, rng, temperature=np.array([0.7, 0.9, 1e-30, 0.5, 1.0, 70_000.0, 0.3, 1.1], np.float32), top_k=0,
               top_p=rng.choice([0.6, 0.99], rows), repetition_penalty=np.array([1.3] * rows, np.float32),
               presence_penalty=0.2, frequency_penalty=0.1)
    g, w = run_both(orc, dev, bits, 0, p, hist, offs, want_probs=False)
    for r in range(rows):
        if r == 5:   # T above 65,536: the 16-bit routes refuse the row
            assert g["tokens"][r] == -1 and g["stats"]["flags"][r] & 0x80000000
            continue
        assert g["tokens"][r] == w["tokens"][r] or exempt_draw(w["margins"][r]), (r, g["tokens"][r], w["tokens"][r])
        assert g["stats"]["flags"][r] == w["stats"]["flags"][r], (r, g["stats"][r], w["stats"][r])


def test_stream_bad_history_tokens_flagged(orc, dev, rng):
    rows, vocab = 4, 5_000
    bits = make_rows(rng, rows, vocab)
    p = params(rows, rng, temperature=1.0, top_k=0, presence_penalty=0.5)
    hist = rng.integers(0, vocab, rows * 100).astype(np.int32)
    hist[5] = -3
    hist[250] = vocab + 10
    offs = np.arange(rows + 1, dtype=np.int64) * 100
    g, w = run_both(orc, dev, bits, 0, p, hist, offs, want_probs=False)
    compare(g, w, p, "badhist")
    assert (g["stats"]["flags"][0] & 16) and (g["stats"]["flags"][2] & 16)


@pytest.mark.parametrize("want_probs", [False, True])
@pytest.mark.parametrize("vocab,length", [(5_000, 100), (5_001, 100), (5_001, 5_000), (500_001, 24_000)])
def test_stream_every_bad_history_token_is_flagged(orc, dev, rng, vocab, length, want_probs):
    """One token outside the vocabulary per row, among valid ones: -1, -2, INT_MIN,
    the first id past the end, INT_MAX; a clean row; over both batch sizes of the
    history view and the one built in the workspace."""
    bad = [-1, -2, -(2 ** 31), vocab, 2 ** 31 - 1, 0]
    rows = len(bad)
    bits = make_rows(rng, rows, vocab)
    p = params(rows, rng, temperature=1.0, top_k=0, presence_penalty=0.5)
    hist = rng.integers(0, vocab, (rows, length)).astype(np.int32)
    hist[np.arange(rows), rng.integers(0, length, rows)] = np.array(bad, np.int64).astype(np.int32)
    offs = np.arange(rows + 1, dtype=np.int64) * length
    g, w = run_both(orc, dev, bits, 0, p, hist.reshape(-1), offs, want_probs=want_probs)
    compare(g, w, p, "badhist")
    assert (g["stats"]["flags"] & 16).astype(bool).tolist() == [True] * 5 + [False]


@pytest.mark.parametrize("dtype", [0, 1, 2])
@pytest.mark.parametrize("want_probs", [False, True])
@pytest.mark.parametrize("vocab", [4_096, 4_099])
def test_stream_min_p_between_weights_closer_than_fp32(orc, dev, rng, dtype, want_probs, vocab):
    """Logits so small, or temperatures so high, that their weights round to one
    another in single precision: min_p 1 keeps the largest ones only, and min_p at
    the weight of a value between two neighbours keeps what lies above."""
    rows = 4
    x = rng.integers(1, 40, (rows, vocab)).astype(np.float32) * np.float32(2.0 ** -10)
    bits = {0: lambda: (x.view(np.uint32) >> 16).astype(np.uint16), 1: lambda: x.astype(np.float16).view(np.uint16),
            2: lambda: x}[dtype]()
    p = params(rows, rng, temperature=np.array([60_000, 60_000, 30_000, 65_536], np.float32), top_p=1.0,
               min_p=np.array([1.0, 1.0 - 2.0 ** -24, 1.0, 1.0 - 2.0 ** -23], np.float32))
    g, w = run_both(orc, dev, bits, dtype, p, want_probs=want_probs)
    assert (w["stats"]["support"][[0, 2]] < vocab // 20).all()
    assert np.array_equal(g["stats"]["support"], w["stats"]["support"]), (g["stats"], w["stats"])
    assert np.array_equal(g["tokens"], w["tokens"])
    if want_probs:
        assert np.array_equal(g["probs"] > 0, w["probs"] > 0)


@pytest.mark.parametrize("dtype", [0, 1, 2])
@pytest.mark.parametrize("vocab", [64, 4_099])
def test_stream_top_p_of_nothing_keeps_the_first_logit(orc, dev, rng, dtype, vocab):
    """top_p so small that its share of the mass is below the sums' unit, 0, or
    negative: the support is the row's first logit (first id among equal ones), alone
    and beside the other filters, with probabilities and without; the same row's
    verification accepts and corrects from that support."""
    import voidinfer_amd as vi
    rows = 8
    bits = make_rows(rng, rows, vocab, std=1.0, dtype=dtype)
    bits[1::2] = 0                                       # all equal: id 0
    p = params(rows, rng, temperature=0.8, top_k=np.array([0, 0, 100, 100, 0, 0, 0, 0]),
               top_p=np.array([0, 0, 0, 0, 1e-14, 1e-14, -0.5, -0.5], np.float32),
               min_p=np.array([0, 0, 0, 0, 0.1, 0.1, 0, 0], np.float32))
    for want_probs in (False, True):
        g, w = run_both(orc, dev, bits, dtype, p, want_probs=want_probs)
        assert (w["stats"]["support"] == 1).all() and (w["tokens"][1::2] == 0).all()
        assert np.array_equal(g["tokens"], w["tokens"]) and np.array_equal(g["stats"]["support"], w["stats"]["support"])
        np.testing.assert_allclose(g["stats"]["support_mass"], 1.0, rtol=1e-6)
        if want_probs:
            assert np.array_equal(g["probs"] > 0, w["probs"] > 0)
    drafted = np.where(np.arange(rows) % 3 == 0, w["tokens"], 1).astype(np.int32)
    t = to_dev(bits, dtype, dev)
    got = vi.verify_rows(vi.VERIFY_SAMPLED, t, torch.from_numpy(drafted).to(dev), rows, 1, draft=t, params=p)
    want = orc.verify_rows(1, bits, dtype, bits, dtype, rows, 1, drafted, p, ())
    for a, b in zip(got, want):
        assert np.array_equal(a, b)


@pytest.mark.parametrize("vocab,length", [(5_001, 4_096), (5_001, 4_097), (5_001, 8_193), (5_001, 16_384),
                                          (5_001, 16_385), (5_001, 40_000), (300_001, 3_200), (300_001, 3_202),
                                          (524_288, 16_256), (524_288, 16_260), (524_287, 70_000)])
def test_stream_history_view_sizes(orc, dev, rng, vocab, length):
    """Histories at the edges of the view's batches and of where its counts lie (half
    a CU's LDS, a CU's, the workspace): tokens seen once and many times, one of them
    up to the whole history, a short and an empty history beside the longest."""
    rows = 5
    bits = make_rows(rng, rows, vocab, std=0.5)
    p = params(rows, rng, temperature=rng.uniform(0.5, 1.2, rows), top_k=0, top_p=0.95,
               repetition_penalty=rng.uniform(1.0, 1.3, rows), presence_penalty=0.2, frequency_penalty=0.001)
    hist = [rng.integers(0, vocab, length), np.tile(rng.choice(vocab, length // 2, replace=length // 2 > vocab), 2),
            np.full(length, vocab - 1), rng.integers(vocab - 40, vocab, 100), np.zeros(0, int)]
    offs = np.concatenate([[0], np.cumsum([len(h) for h in hist])]).astype(np.int64)
    stream(orc, dev, bits, 0, p, np.concatenate(hist).astype(np.int32), offs, f"view-{vocab}-{length}")


def test_stream_repeat_calls_same_workspace(orc, dev, rng):
    """The part and arrival counters reset themselves: three calls in a row
    on one workspace give the same outputs."""
    import voidinfer_amd as vi
    rows, vocab = 24, 248_320
    bits = make_rows(rng, rows, vocab, std=1.0)
    p = params(rows, rng, temperature=rng.uniform(0.5, 1.2, rows), top_k=0, top_p=0.9)
    t = to_dev(bits, 0, dev)
    outs = []
    for i in range(3):
        print(f"[stream] repeat call {i}", flush=True)
        o = vi.sample_rows(t, p, want_probs=False)
        torch.cuda.synchronize()
        outs.append((o.tokens.cpu().numpy(), vi.stats_numpy(o.stats)))
    for tok, st in outs[1:]:
        assert np.array_equal(tok, outs[0][0])
        assert np.array_equal(st, outs[0][1])
    w_tok, _, _, _, margins = orc.sample_rows(bits, 0, p, None, None, want_probs=False)
    for r in range(rows):
        assert outs[0][0][r] == w_tok[r] or exempt_draw(margins[r]), r


@pytest.mark.parametrize("dtype", [0, 1])
def test_stream_state_route_steps(orc, dev, rng, dtype):
    """Penalties from penalty states over decode steps; odd steps record the
    sampled tokens in the same launch.  Every step against the oracle over the
    equivalent history."""
    import voidinfer_amd as vi
    from voidinfer_amd import workloads as W
    rows, vocab, L = 12, 248_320, 6000
    x = W.gaussian_zipf(rows, vocab, 1.0, int(rng.integers(1 << 30)))
    bits = W.encode(x, {0: "bf16", 1: "f16"}[dtype])
    p = vi.params_array(rows, seed=rng.integers(1, 2**62, rows), position=rng.integers(0, 10**5, rows),
                        temperature=rng.uniform(0.5, 1.2, rows), top_k=np.array([0, 0, 100, 0, 1000, 0] * 2),
                        top_p=rng.choice([0.9, 0.95, 1.0], rows), min_p=rng.choice([0.0, 0.02], rows),
                        repetition_penalty=rng.uniform(1.0, 1.3, rows), presence_penalty=rng.uniform(0, 0.5, rows),
                        frequency_penalty=rng.uniform(0.0, 0.3, rows))
    hist = []
    for r in range(rows):
        top = np.argsort(-x[r])[:300]                # penalties that reorder the top candidates
        h = np.concatenate([rng.integers(0, vocab, L), rng.choice(top, 800), np.repeat(top[:5], 40)])
        hist.append(rng.permutation(h).astype(np.int32))
    st = vi.PenaltyState(rows, vocab, 1 << 14, device=dev)
    toks, offs = np.concatenate(hist), np.concatenate([[0], np.cumsum([len(h) for h in hist])]).astype(np.int64)
    st.update(torch.from_numpy(toks).to(dev), torch.from_numpy(offs).to(dev))
    logits = to_dev(bits, dtype, dev)
    for step in range(4):
        print(f"[stream] state dtype={dtype} step={step}", flush=True)
        fused = step % 2 == 1
        b = vi.sample_rows_state(logits, p, st, record=fused, want_probs=False)
        torch.cuda.synchronize()
        toks = np.concatenate(hist)
        offs = np.concatenate([[0], np.cumsum([len(h) for h in hist])]).astype(np.int64)
        w_tok, w_u, _, w_stats, margins = orc.sample_rows(bits, dtype, p, toks, offs, want_probs=False)
        g_tok = b.tokens.cpu().numpy()
        g_st = vi.stats_numpy(b.stats)
        for r in range(rows):
            if g_tok[r] != w_tok[r] or g_st["support"][r] != w_stats["support"][r]:
                assert exempt_draw(margins[r]), (step, r, g_tok[r], w_tok[r], g_st[r], w_stats[r], margins[r])
        if not fused:
            st.update(b.tokens)
        hist = [np.append(h, t).astype(np.int32) for h, t in zip(hist, g_tok)]
        p["position"] += 1


def test_stream_config5_all_rows(orc, dev):
    """Configuration 5 at full size (128 rows, 32,768-token histories): the
    state route (as the benchmark runs it) and the history route."""
    import voidinfer_amd as vi
    from voidinfer_amd import workloads as W
    bits, hist, offs, p = W.config5()
    st = vi.PenaltyState(128, W.V_QWEN, 1 << 16, device=dev)
    st.update(torch.from_numpy(hist).to(dev), torch.from_numpy(offs).to(dev))
    logits = to_dev(bits, 0, dev)
    print("[stream] config5 state route", flush=True)
    b = vi.sample_rows_state(logits, p, st, want_probs=False)
    print("[stream] config5 history route", flush=True)
    a = vi.sample_rows(logits, p, torch.from_numpy(hist).to(dev), torch.from_numpy(offs).to(dev),
                       max_history=32768, want_probs=False)
    torch.cuda.synchronize()
    w_tok, w_u, _, w_stats, margins = orc.sample_rows(bits, 0, p, hist, offs, want_probs=False)
    for name, o in (("state", b), ("history", a)):
        g_tok = o.tokens.cpu().numpy()
        g_st = vi.stats_numpy(o.stats)
        exempt = 0
        for r in range(128):
            if g_tok[r] != w_tok[r] or g_st["support"][r] != w_stats["support"][r]:
                assert exempt_draw(margins[r]), (name, r, g_tok[r], w_tok[r], g_st[r], w_stats[r], margins[r])
                exempt += 1
                continue
            assert g_st["flags"][r] == w_stats["flags"][r] and g_st["finite"][r] == w_stats["finite"][r], (name, r)
            np.testing.assert_allclose(g_st["support_mass"][r], w_stats["support_mass"][r], rtol=1e-6)
        assert exempt <= 2, (name, exempt)


@pytest.mark.parametrize("dtype", [0, 1])
@pytest.mark.parametrize("rows,vocab", [(3, 200_000), (9, 24_576 * 4 + 8), (1, 12_288 * 2)])
def test_stream_many_groups_and_top_key(orc, dev, rng, dtype, rows, vocab):
    """Rows whose logits spread over every exponent (more occupied groups than
    the merge keeps), and rows whose largest valid key is hard to find: negative
    logits only, signed zeros only, the highest groups holding nothing valid."""
    x = rng.standard_normal((9, vocab)).astype(np.float32) * np.exp2(rng.uniform(-14, 4, (9, vocab))).astype(np.float32)
    x[1] = -np.abs(x[1]) - np.float32(1e-3)
    x[2] = np.where(rng.random(vocab) < 0.5, 0.0, -0.0)
    x[3] = np.where(rng.random(vocab) < 0.9, -np.abs(x[3]), -0.0)
    bits = x.astype(np.float16).view(np.uint16) if dtype else (x.view(np.uint32) >> 16).astype(np.uint16)
    inf_ = 0x7C00 if dtype else 0x7F80
    big = 0x7BFF if dtype else 0x7F00
    bits[1, ::9] = inf_                                  # nothing valid above the negative keys
    bits[4, ::5] = big                                   # finite patterns whose z overflows (T 1e-36)
    bits[4, 3] = inf_ + 1
    bits = bits[:rows] if rows > 1 else bits[4:5]
    t = np.array([0.7, 0.9, 1.0, 0.5, 1e-36, 0.8, 1.2, 0.6, 0.7], np.float32)
    p = params(rows, rng, temperature=t[:rows] if rows > 1 else t[4:5], top_k=rng.choice([0, 0, 300], rows),
               top_p=rng.choice([0.9, 0.95, 1.0], rows), min_p=rng.choice([0.0, 0.01], rows))
    stream(orc, dev, np.ascontiguousarray(bits), dtype, p, label=f"groups-{dtype}-{rows}-{vocab}")


@pytest.mark.parametrize("dtype", [0, 1])
@pytest.mark.parametrize("vocab", [1, 7, 13, 4_099, 65_505, 131_015, 500_001])
def test_stream_odd_rows_and_probabilities(orc, dev, rng, dtype, vocab):
    """Rows off a 16-byte boundary, logits past the last whole vector (a last part
    of one logit at 65,505), supports that cut the logits of their last key, the
    distribution's tokens seen once and more than once; at 500,001 tokens the
    history view's bitmaps and counts exceed the LDS."""
    rows, L = 9, 24_000 if vocab > 400_000 else 600
    bits = make_rows(rng, rows, vocab, std=1.0, dtype=dtype)
    bits[1::4] &= 0xFFC0 if dtype == 0 else 0xFE00        # few values: many ties at every cut
    bits[2, -1] = bits[2].max() if vocab < 8 else 0x4380   # the row's last logit is drawn
    p = params(rows, rng, temperature=rng.uniform(0.5, 1.2, rows), top_k=rng.choice([0, 70, 1000], rows),
               top_p=rng.choice([0.8, 0.95, 1.0], rows), min_p=rng.choice([0.0, 0.0, 0.02], rows),
               repetition_penalty=rng.uniform(1.0, 1.2, rows), presence_penalty=0.1, frequency_penalty=0.03)
    p["repetition_penalty"][3], p["presence_penalty"][3], p["frequency_penalty"][3] = 1.0, 0.0, 0.0
    hist = rng.integers(0, vocab, (rows, L)).astype(np.int32)
    hist[:, :40] = rng.integers(max(0, vocab - 9), vocab, (rows, 40))   # the tail's tokens, repeated
    offs = np.arange(rows + 1, dtype=np.int64) * L
    compare(*run_both(orc, dev, bits, dtype, p, hist.reshape(-1), offs, want_probs=True), p, f"odd-{dtype}-{vocab}")


def test_stream_more_rows_than_one_launch(orc, dev, rng):
    """32,777 rows: two launches over the same tables, the second of nine rows."""
    import voidinfer_amd as vi
    rows, vocab = 32_777, 40
    bits = make_rows(rng, 64, vocab, std=1.0)[np.arange(rows) % 64]
    p = params(rows, rng, temperature=0.8, top_k=0, top_p=0.9)
    out = vi.sample_rows(to_dev(bits, 0, dev), p, want_probs=True)
    torch.cuda.synchronize()
    at = np.array([0, 1, 8_191, 32_767, 32_768, 32_769, 32_776])
    g = dict(tokens=out.tokens.cpu().numpy()[at], u=out.uniforms.cpu().numpy()[at], probs=out.probs.cpu().numpy()[at],
             stats=vi.stats_numpy(out.stats)[at])
    tok, u, probs, stats, margins = orc.sample_rows(bits[at], 0, p[at], None, None, want_probs=True)
    compare(g, dict(tokens=tok, u=u, probs=probs, stats=stats, margins=margins), p[at], "rows")
