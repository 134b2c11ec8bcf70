"""Room for filter records: long motifs and lowercase bases leave the default
form more than one record per hit, which callers that state their hits need not
know (needs the GPU)."""
from __future__ import annotations

import numpy as np
import pytest

import blamm_amd as ba
from blamm_amd import synth
from helpers import library, stream_case

pytestmark = pytest.mark.gpu


def workload(lmin, lmax, lower_every, n=1_500_000):
    text, runs, bg = stream_case(lmin + lower_every, n, lower_every=lower_every)
    pwms, thr = library(synth.motifs(120, lmin, lmax, 0.4, seed=lmax), bg, pvalue=1e-3)
    P, lengths, _ = ba.build_pattern_matrix(pwms)
    packed, lower = ba.pack(text)
    return P, lengths, thr, packed, lower, len(text), runs


@pytest.mark.parametrize("lmin,lmax,lower_every", [(24, 60, 0), (6, 25, 400)])
def test_batches_run_once_with_exact_expectations(lmin, lmax, lower_every):
    """Batches whose request states the number of its hits do not grow their
    buffers and run again, and have the scan's hits: one of 81 % of a stream,
    then one of the whole (which has 1.5 times its hits of room from the first)."""
    P, lengths, thr, packed, lower, n, runs = workload(lmin, lmax, lower_every)
    with ba.HipScanner(0) as sc:
        sc.set_library(P, lengths, thr, ba.PREC_BF16X2)
        b = ba.Batch(sc, max_bases=n + 64, max_requests=1)
        try:
            for m in (81 * n // 100, n):
                starts = [r for r in runs if r < m]
                want = np.sort(sc.scan(packed, m, starts, lower), order=["pos", "col"])
                assert len(want) > 200_000
                b.submit([ba.ScanRequest(packed, m, starts, lower, None, len(want))])
                before = b.device_bytes()
                assert b.wait() == len(want)
                assert b.device_bytes() == before
                assert np.array_equal(np.sort(b.hits(0), order=["pos", "col"]), want)
        finally:
            b.close()


@pytest.mark.parametrize("lmin,lmax,lower_every", [(24, 60, 0), (6, 25, 400)])
def test_reserve_holds_a_record_per_score(lmin, lmax, lower_every):
    """Room reserved for the records of a filter by scores (those of the
    split-BF16 form, and a tenth more) is enough for the default form's first
    scan."""
    import torch
    P, lengths, thr, packed, lower, n, runs = workload(lmin, lmax, lower_every)
    records = 0
    for prec in (ba.PREC_BF16X2_LO, ba.PREC_BF16X2):
        with ba.HipScanner(0) as sc:
            sc.set_library(P, lengths, thr, prec)
            if records:
                sc.reserve(int(1.1 * records))
            else:
                sc.reserve(1 << 23)
            words = np.zeros(int(sc.lib.blamm_hip_packed_words(n)), np.uint64)
            words[:packed.size] = packed
            mask = None
            if lower is not None:
                mask = np.zeros(int(sc.lib.blamm_hip_mask_words(n)), np.uint64)
                mask[:lower.size] = lower
                mask = torch.from_numpy(mask.view(np.int64)).to("cuda:0")
            words = torch.from_numpy(words.view(np.int64)).to("cuda:0")
            starts = torch.from_numpy(np.asarray(runs, np.uint64).view(np.int64)).to("cuda:0")
            hits = torch.zeros(1 << 23, dtype=torch.int64, device="cuda:0")
            torch.cuda.synchronize()
            sc.scan_device(words, mask, n, starts, len(runs), hits, 1 << 22, None)
            assert sc.scan_finish() > 200_000
            records = sc.stats().candidates


def test_server_counts_the_second_record():
    """Two requests that would fill a slot's budget with one record per
    expected hit are not put into one batch; each alone is accepted."""
    P, lengths, thr, packed, lower, n, runs = workload(6, 25, 0, n=200_000)
    with ba.HipScanner(0) as sc:
        sc.set_library(P, lengths, thr, ba.PREC_BF16X2)
        srv = ba.Server(sc, hbm_budget_bytes=100_000_000, slots=1)
        try:
            ids = [srv.submit(ba.ScanRequest(packed, n, runs, lower, None, 1_000_000)) for _ in range(6)]
            for i in ids:
                assert srv.wait(i, 60_000)
                assert srv.release(i).batch_requests == 1
        finally:
            srv.close()


def lowercase_bound(w, weight):
    """What the screen's bound of an all lowercase window of column w is above 0,
    in weights: its layout for masked streams restated, with the slack of a
    lowercase base counted `weight` times that of an uppercase one."""
    def fp6(x, rounded):
        m = np.abs(x)
        step = np.where(m < 2, 0.125, np.where(m < 4, 0.25, 0.5))
        return np.clip(rounded(x / step) * step, -7.5, 7.5)

    w = w.astype(np.float64)
    alpha = 7.5 / np.abs(w).max()
    pi = 2.0 ** np.maximum(w - w.max(1, keepdims=True), -60)
    pi /= pi.sum(1, keepdims=True)
    slack, excess = [], []
    for rounded in (np.rint, np.ceil):
        y = fp6(alpha * w, rounded)
        e = np.maximum(0.0, (alpha * w - y).max(1))
        excess.append(e)
        slack.append((pi * (e[:, None] + y - alpha * w)).sum(1) + weight * e)
    return np.where(slack[1] < slack[0], excess[1], excess[0]).sum() / alpha


def test_lowercase_windows_above_their_bound_leave_no_records():
    """Lowercase windows score 0.  A long column's threshold need be 0.3 to 1.2
    bits above that for the default form to rule them out, and 0.5 to 1 bit more
    if the slack of lowercase bases did not count where weights are rounded."""
    text, runs, bg = stream_case(8, 20_000)
    pwms, _ = library(synth.motifs(60, 50, 60, 0.4, seed=8), bg, pvalue=1e-4)
    thr = np.array([lowercase_bound(w, 1.0) for w in pwms]) + 0.15
    assert np.min([lowercase_bound(w, 0.0) for w in pwms] - thr) > 0.2
    text = (np.frombuffer(text, np.uint8) | 0x20).tobytes()
    packed, lower = ba.pack(text)
    P, lengths, _ = ba.build_pattern_matrix(pwms)
    with ba.HipScanner(0) as sc:
        sc.set_library(P, lengths, thr.astype(np.float32), ba.PREC_BF16X2)
        sc.scan(packed, len(text), runs, lower)
        # two records at most of each of the tiles whose windows reach the
        # padding, which is not lowercase: 59 windows and the last tile's rest
        assert sc.stats().candidates <= 2 * 4 * len(pwms)
