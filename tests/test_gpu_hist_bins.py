"""Binning of empirical histograms at its edges, count for count against the
oracle: bin numbers around the LDS variant's limit, ranges that scores leave or
do not reach, columns whose bins are narrower than the score margins, and many
windows next to a bin edge."""
from __future__ import annotations

import numpy as np
import pytest

import blamm_amd as ba
from blamm_amd import synth

pytestmark = pytest.mark.gpu


def inputs(seed, n, lengths, lower=0.0):
    rng = np.random.default_rng(seed)
    codes = rng.integers(0, 4, size=n).astype(np.uint8)
    text = synth.CODE2BASE[codes].copy()
    if lower:
        text[rng.random(n) < lower] |= 0x20
    runs = np.unique(np.concatenate([[0], rng.integers(0, n, size=max(1, n // 500))])).astype(np.uint64)
    pwms = [rng.normal(-0.5, 2.0, size=(L, 4)).astype(np.float32) for L in lengths]
    return text.tobytes(), runs, pwms


def check(text, runs, pwms, mn, mx, nbins):
    import oracle
    mn, mx = np.asarray(mn, np.float32), np.asarray(mx, np.float32)
    P, lengths, _ = ba.build_pattern_matrix(pwms)
    packed, lower = ba.pack(text)
    with ba.HipScanner(0) as sc:
        sc.set_library(P, lengths, np.zeros(len(pwms), np.float32), ba.PREC_BF16X2)
        got = sc.hist(packed, len(text), mn, mx, nbins, runs, lower)
    want = oracle.empirical_hist(text, runs, pwms, mn, mx, nbins, threads=4)
    assert np.array_equal(got, want)
    return got


def ranges(pwms):
    return [ba.min_score(w) for w in pwms], [ba.max_score(w) for w in pwms]


@pytest.mark.parametrize("lower", [0.0, 0.3])
@pytest.mark.parametrize("nbins", [1, 2, 250, 511, 512, 513])
def test_bin_counts(nbins, lower):
    text, runs, pwms = inputs(nbins, 20_011, list(range(1, 33)) + [33, 48, 64], lower)
    check(text, runs, pwms, *ranges(pwms), nbins)


@pytest.mark.parametrize("case", ["inside", "below", "above", "far", "tiny", "zero", "wide"])
def test_ranges(case):
    """Ranges that are not the columns' own: scores outside go to the first
    and last bin."""
    text, runs, pwms = inputs(len(case), 12_001, [5, 8, 12, 17, 20, 31, 40], 0.1)
    mn, mx = (np.asarray(v, np.float64) for v in ranges(pwms))
    mid, half = (mn + mx) / 2, (mx - mn) / 2
    lo, hi = {"inside": (mid - 0.2 * half, mid + 0.2 * half), "below": (mn - 3 * half, mid), "above": (mid, mx + 3 * half),
              "far": (mx + 1e5, mx + 1e5 + half), "tiny": (mid, mid + 1e-4), "zero": (mid, mid),
              "wide": (mn - 1e6, mx + 1e6)}[case]
    check(text, runs, pwms, lo, hi, 250)


def test_scores_on_bin_edges():
    """Whole weights and whole bins: every window lies on an edge."""
    text, runs, pwms = inputs(5, 30_000, [6] * 40 + [18] * 30)
    pwms = [np.rint(w) for w in pwms]
    mn, mx = ranges(pwms)
    for nbins in (64, 128):
        got = check(text, runs, pwms, mn, [a + nbins for a in mn], nbins)
    assert got.sum() > 0


@pytest.mark.parametrize("longest", [24, 40])
@pytest.mark.parametrize("lower", [0.0, 0.3])
@pytest.mark.parametrize("nbins", [1, 250, 512, 513])
def test_scores_beyond_fp32(nbins, lower, longest):
    """Finite weights whose sums overflow FP32, beside ordinary columns: an
    infinite score has no bin coordinate and is counted in the first bin, as
    int() of the reference's quotient gives it; the same for a width of zero
    and for a minimum so low that the distance from it overflows."""
    text, runs, pwms = inputs(nbins + 7, 9_001, [2, 2, 2, 6, 9, longest, 12, 5], lower)
    mn, mx = (np.asarray(v, np.float64) for v in ranges(pwms))
    big = 2e38
    pwms[0] = np.array([[big, -big, 1, 0], [big, -big, 0, 1]], np.float32)
    mn[0], mx[0] = 0.0, 3e38
    pwms[1] = pwms[0].copy()
    mn[1] = mx[1] = 1.0
    pwms[2] = np.array([[3.4e38, -3.4e38, 1e38, 0], [1, 0, 2, 3]], np.float32)     # bf16 rounds these to infinity
    mn[2], mx[2] = -1e38, 2e38
    pwms[3][0, 1] = 2e38
    mn[3], mx[3] = -2.5e38, 0.5e38
    pwms[5] = (pwms[5] * 1e37).astype(np.float32)
    mn[5], mx[5] = -3e37, 2e38
    with np.errstate(over="ignore"):
        got = check(text, runs, pwms, mn, mx, nbins)
    assert got[:3, 0].min() > 0


@pytest.mark.parametrize("n", [1, 33, 511, 513, 2_049, 70_001])
@pytest.mark.parametrize("columns", [3, 70])
def test_small_calls(n, columns):
    """Calls of one work item and of many short ones."""
    text, runs, pwms = inputs(n, n, [6 + i % 19 for i in range(columns)])
    check(text, runs, pwms, *ranges(pwms), 250)
