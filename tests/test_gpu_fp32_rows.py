"""The FP32 form's three products per position (streams without lowercase
bases): hit sets against the FP64 oracle at every chunk count, at the stream's
edges, for weights whose differences leave FP32's range, and in batches."""
from __future__ import annotations

import numpy as np
import pytest

import blamm_amd as ba
from test_gpu_screen import check, random_pwms, stream, thresholds

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("lower", [0.0, 0.3])
@pytest.mark.parametrize("ncols", [1, 15, 17, 70])
def test_every_length(ncols, lower):
    """Every chunk count from 1 to 16 and every remainder of four positions."""
    for lo in range(1, 65, 16):
        rng = np.random.default_rng([ncols, lo])
        pwms = random_pwms(rng, [lo + i % 16 for i in range(ncols)])
        text, runs = stream(rng, 1501, lower)
        check(pwms, thresholds(pwms, 0.45), text, runs, ba.PREC_FP32)


@pytest.mark.parametrize("n", [1, 16, 31, 33, 64, 65, 1023])
def test_stream_edges(n):
    rng = np.random.default_rng(n)
    pwms = random_pwms(rng, rng.integers(1, 40, size=70))
    text, runs = stream(rng, n, 0.0)
    check(pwms, thresholds(pwms, 0.3), text, runs, ba.PREC_FP32)


@pytest.mark.parametrize("case", ["tiny", "mixed", "ties", "far_constant", "out_of_range"])
def test_weights_of_any_scale(case):
    rng = np.random.default_rng(len(case))
    lengths = rng.integers(1, 33, size=48)
    pwms = random_pwms(rng, lengths, 1e-30 if case == "tiny" else 1.0)
    if case == "mixed":
        pwms = [(w * 10.0 ** rng.uniform(-6, 6, size=(w.shape[0], 1))).astype(np.float32) for w in pwms]
    elif case == "ties":            # whole scores on whole thresholds
        pwms = [np.where(w == w.max(1, keepdims=True), 1.0, 0.0).astype(np.float32) for w in pwms]
    elif case == "far_constant":    # the last base far from the others
        for w in pwms:
            w[:, 3] = -1.0e7
    elif case == "out_of_range":    # differences, or their sums, beyond FP32
        for i, w in enumerate(pwms):
            if i % 3 == 0:
                w[0] = [3.0e38, 1.0, -1.0, -3.0e38]
            elif i % 3 == 1:
                w[:, 0] = -3.0e37
    thr = thresholds(pwms, 0.4)
    if case == "ties":
        thr = np.array([np.ceil(0.5 * w.shape[0]) for w in pwms], np.float32)
    elif case == "far_constant":
        thr = np.array([0.4 * w[:, :3].max(1).sum(dtype=np.float64) for w in pwms], np.float32)
    elif case == "out_of_range":
        thr = np.array([1.0e38 if i % 3 == 0 else 0.3 * w[:, 1:].max(1).sum(dtype=np.float64)
                        for i, w in enumerate(pwms)], np.float32)
    text, runs = stream(rng, 1500, 0.0)
    check(pwms, thr, text, runs, ba.PREC_FP32)


@pytest.mark.parametrize("lower", [0.0, 0.2])
def test_batch_matches_single_scans(lower):
    rng = np.random.default_rng(78)
    pwms = random_pwms(rng, rng.integers(1, 64, size=90))
    thr = thresholds(pwms, 0.45)
    P, lengths, _ = ba.build_pattern_matrix(pwms)
    with ba.HipScanner(0) as sc:
        sc.set_library(P, lengths, thr, ba.PREC_FP32)
        reqs, want = [], []
        for r in range(5):
            text, runs = stream(rng, int(rng.integers(1, 3000)), lower)
            packed, low = ba.pack(text)
            t = np.where(rng.random(len(pwms)) < 0.6, thr, np.float32(np.inf)).astype(np.float32)
            reqs.append(ba.ScanRequest(packed, len(text), runs, low, t))
            h = sc.scan(packed, len(text), runs, low)
            want.append(np.sort(h[np.isfinite(t[h["col"]])], order=["pos", "col"]))
        b = ba.Batch(sc, max_bases=20_000, max_requests=5)
        b.submit(reqs)
        b.wait()
        for r in range(5):
            assert np.array_equal(np.sort(b.hits(r), order=["pos", "col"]), want[r])
        b.close()
