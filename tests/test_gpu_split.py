"""The split-BF16 form behind the screen: hit sets against the FP64 oracle at
every number of steps, around the 64 tiles that a wave marks at once, with few
and with all tile blocks marked, and in batches."""
from __future__ import annotations

import numpy as np
import pytest

import blamm_amd as ba
from test_gpu_screen import check, random_pwms, stream, thresholds

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("lower", [0.0, 0.3])
@pytest.mark.parametrize("lengths", [[1], [16, 17, 32, 33, 48, 49, 64], [12] * 257 + [20] * 129 + [40] * 65 + [60] * 33],
                         ids=["one", "every_step", "groups"])
def test_lengths_and_groups(lengths, lower):
    rng = np.random.default_rng([len(lengths), int(10 * lower)])
    pwms = random_pwms(rng, lengths)
    text, runs = stream(rng, 3001, lower)
    check(pwms, thresholds(pwms, 0.45), text, runs, ba.PREC_BF16X2_LO)


@pytest.mark.parametrize("tiles", [1, 63, 64, 65, 129])
@pytest.mark.parametrize("share", [0.7, -10.0])
def test_marked_tiles(tiles, share):
    rng = np.random.default_rng(tiles)
    pwms = random_pwms(rng, rng.integers(4, 40, size=40))
    text, runs = stream(rng, 32 * tiles, 0.0)
    check(pwms, thresholds(pwms, share), text, runs, ba.PREC_BF16X2_LO, (512, 2, 4))


@pytest.mark.parametrize("lower", [0.0, 0.2])
def test_batch_matches_single_scans(lower):
    rng = np.random.default_rng(79)
    pwms = random_pwms(rng, rng.integers(1, 64, size=90))
    thr = thresholds(pwms, 0.45)
    P, lengths, _ = ba.build_pattern_matrix(pwms)
    with ba.HipScanner(0) as sc:
        sc.set_library(P, lengths, thr, ba.PREC_BF16X2_LO)
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
