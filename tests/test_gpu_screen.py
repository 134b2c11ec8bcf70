"""The screen of the default form (integer upper bounds on FP6 x FP4 tiles) and
the filters' work queues: hit sets against the FP64 oracle at the edges of
steps, blocks, groups, tiles and items, and for weights of any scale."""
from __future__ import annotations

import numpy as np
import pytest

import blamm_amd as ba
from blamm_amd import synth

pytestmark = pytest.mark.gpu


def random_pwms(rng, lengths, scale=1.0, spread=3.0):
    return [(scale * rng.normal(0.0, spread, size=(L, 4)) - scale).astype(np.float32) for L in lengths]


def stream(rng, n, lower):
    codes = rng.integers(0, 4, size=n).astype(np.uint8)
    text = synth.CODE2BASE[codes].copy()
    if lower:
        text[rng.random(n) < lower] |= 0x20
    runs = np.unique(np.concatenate([[0], rng.integers(0, n, size=max(1, n // 400))])).astype(np.uint64)
    return text.tobytes(), runs


def thresholds(pwms, share):
    """A share of the way from the mean to the best score of each column."""
    best = np.array([w.max(1).sum(dtype=np.float64) for w in pwms])
    mean = np.array([w.mean(1).sum(dtype=np.float64) for w in pwms])
    return (mean + share * (best - mean)).astype(np.float32)


def check(pwms, thr, text, runs, precision=ba.PREC_BF16X2, tuning=None):
    import oracle
    P, lengths, _ = ba.build_pattern_matrix(pwms)
    packed, lower = ba.pack(text)
    ref = oracle.scan_fp64(text, runs, pwms, thr)
    want = set(zip(ref["pos"].tolist(), ref["col"].tolist()))
    with ba.HipScanner(0) as sc:
        if tuning:
            sc.set_tuning(*tuning)
        sc.set_library(P, lengths, np.asarray(thr, np.float32), precision)
        h = sc.scan(packed, len(text), runs, lower)
    assert len(h) == len(want)
    assert set(zip(h["pos"].tolist(), h["col"].tolist())) == want
    return len(want)


@pytest.mark.parametrize("lower", [0.0, 0.3])
@pytest.mark.parametrize("lengths", [
    [1], [15, 16, 17], [31, 32, 33], [47, 48, 49, 63, 64], [1, 16, 17, 32, 33, 48, 49, 64],
    [8] * 31, [16] * 32, [17] * 33, [12] * 257 + [20] * 129 + [40] * 65 + [60] * 33,
], ids=["one", "step", "two_steps", "long", "every_step", "block-1", "block", "block+1", "groups"])
def test_lengths_and_groups(lengths, lower):
    rng = np.random.default_rng([len(lengths), lengths[0], int(10 * lower)])
    pwms = random_pwms(rng, lengths)
    text, runs = stream(rng, 3001, lower)
    check(pwms, thresholds(pwms, 0.45), text, runs)


@pytest.mark.parametrize("n", [1, 31, 32, 33, 63, 64, 65, 511, 2049])
def test_stream_edges(n):
    rng = np.random.default_rng(n)
    pwms = random_pwms(rng, rng.integers(1, 40, size=70))
    text, runs = stream(rng, n, 0.1 if n % 2 else 0.0)
    check(pwms, thresholds(pwms, 0.3), text, runs)


@pytest.mark.parametrize("lower", [0.0, 0.2])
@pytest.mark.parametrize("case", ["tiny", "huge", "mixed", "constant", "one_hot", "all_pass", "none_pass"])
def test_weights_of_any_scale(case, lower):
    rng = np.random.default_rng(len(case))
    lengths = rng.integers(1, 33, size=48)
    pwms = random_pwms(rng, lengths, {"tiny": 1e-30, "huge": 1e30}.get(case, 1.0))
    share = 0.4
    if case == "mixed":        # columns, positions and bases of very different size
        pwms = [(w * 10.0 ** rng.uniform(-6, 6, size=(w.shape[0], 1))).astype(np.float32) for w in pwms]
    elif case == "constant":   # nothing to tell the bases apart
        pwms = [np.repeat(w[:, :1], 4, axis=1) for w in pwms]
    elif case == "one_hot":
        pwms = [np.where(w == w.max(1, keepdims=True), 1.0, 0.0).astype(np.float32) for w in pwms]
    text, runs = stream(rng, 1500, lower)
    thr = thresholds(pwms, share)
    if case == "constant":     # exactly the score of every window
        thr = np.array([w[:, 0].sum(dtype=np.float64) for w in pwms], np.float32)
    elif case == "one_hot":    # ties: whole scores on whole thresholds
        thr = np.array([np.ceil(0.5 * w.shape[0]) for w in pwms], np.float32)
    elif case == "all_pass":
        thr = np.full(len(pwms), -np.inf, np.float32)
        thr[::5] = -3.0e38
    elif case == "none_pass":
        thr = np.full(len(pwms), np.inf, np.float32)
        thr[::5] = 3.0e38
    check(pwms, thr, text, runs)


@pytest.mark.parametrize("precision", [ba.PREC_BF16X2, ba.PREC_BF16X2_LO, ba.PREC_FP32])
@pytest.mark.parametrize("window", [1, 3, 512])
def test_items_cover_the_stream_once(window, precision):
    """Work items from one tile up, more of them than waves: every item is
    done, and none twice (a hit found twice would show in the hit count)."""
    rng = np.random.default_rng(window)
    pwms = random_pwms(rng, rng.integers(4, 30, size=130))
    text, runs = stream(rng, 200_003, 0.0)
    assert check(pwms, thresholds(pwms, 0.6), text, runs, precision, (window, 1, 4)) > 0


def test_batch_matches_single_scans():
    """Requests with column subsets, with and without lowercase bases, get in a
    batch what a scan of their own gives (gathered screen fragments)."""
    rng = np.random.default_rng(77)
    pwms = random_pwms(rng, rng.integers(1, 64, size=150))
    thr = thresholds(pwms, 0.45)
    P, lengths, _ = ba.build_pattern_matrix(pwms)
    with ba.HipScanner(0) as sc:
        sc.set_library(P, lengths, thr, ba.PREC_BF16X2)
        for lower in (0.0, 0.2):
            reqs, want = [], []
            for r in range(5):
                text, runs = stream(rng, int(rng.integers(1, 3000)), lower)
                packed, low = ba.pack(text)
                t = np.where(rng.random(len(pwms)) < 0.6, thr, np.float32(np.inf)).astype(np.float32)
                reqs.append(ba.ScanRequest(packed, len(text), runs, low, t))
                h = sc.scan(packed, len(text), runs, low)
                h = h[np.isfinite(t[h["col"]])]
                want.append(np.sort(h, order=["pos", "col"]))
            b = ba.Batch(sc, max_bases=20_000, max_requests=5)
            b.submit(reqs)
            b.wait()
            for r in range(5):
                got = np.sort(b.hits(r), order=["pos", "col"])
                assert np.array_equal(got, want[r])
            b.close()
