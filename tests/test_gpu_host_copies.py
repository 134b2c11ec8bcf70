"""Host buffers in and out: streams in any form give the hits of a plain
array, and hits split over threads are the hits of one."""
from __future__ import annotations

import ctypes
import mmap

import numpy as np
import pytest

import blamm_amd as ba
from test_gpu_screen import random_pwms, stream, thresholds

pytestmark = pytest.mark.gpu


def scanner(rng, share):
    pwms = random_pwms(rng, rng.integers(4, 20, size=40))
    P, lengths, _ = ba.build_pattern_matrix(pwms)
    sc = ba.HipScanner(0)
    sc.set_library(P, lengths, thresholds(pwms, share), ba.PREC_BF16X2)
    return sc


def by_place(h):
    return np.sort(h, order=["pos", "col"])


@pytest.mark.parametrize("form", ["longer", "strided", "int64", "list", "shorter", "offset"])
@pytest.mark.parametrize("n", [1, 31, 2001])
def test_stream_forms(form, n):
    rng = np.random.default_rng(n)
    text, runs = stream(rng, n, 0.2)
    codes, lower = ba.pack(text)
    if lower is None:
        lower = np.zeros(1, np.uint64)
    with scanner(rng, 0.3) as sc:
        need = [(n + 31) // 32, (n + 63) // 64]
        plain = [np.concatenate([a, np.zeros(16, np.uint64)])[:k + 16] for a, k in zip((codes, lower), need)]
        want = by_place(sc.scan(plain[0], n, runs, plain[1]))

        def as_form(a, k):
            if form == "longer":
                return np.concatenate([a[:k], np.full(99, ~np.uint64(0))])
            if form == "strided":
                return np.repeat(a[:k], 2)[::2]
            if form == "int64":
                return a[:k].view(np.int64).copy()
            if form == "list":
                return [int(x) for x in a[:k]]
            if form == "offset":
                return np.frombuffer(b"\0" + a[:k].tobytes(), np.uint8)[1:].view(np.uint64)
            return np.trim_zeros(a[:k], "b")

        c, low = as_form(plain[0], need[0]), as_form(plain[1], need[1])
        assert np.array_equal(by_place(sc.scan(c, n, runs, low)), want)
        assert np.array_equal(by_place(sc.scan_pinned(c, n, runs, low)), want)


@pytest.mark.parametrize("n", [40_000, 150_001])
def test_many_hits(n):
    """More hits than one thread copies, in the three ways they come back."""
    rng = np.random.default_rng(n)
    text, runs = stream(rng, n, 0.0)
    codes, _ = ba.pack(text)
    with scanner(rng, 0.0) as sc:
        want = by_place(sc.scan(codes, n, runs))
        assert len(want) > 16 * 32768
        assert np.array_equal(by_place(sc.scan_pinned(codes, n, runs)), want)
        b = ba.Batch(sc, max_bases=2 * n + 4096, max_requests=3)
        b.submit([ba.ScanRequest(codes, n, runs), ba.ScanRequest(codes[:1], 20, runs[:1]),
                  ba.ScanRequest(codes, n, runs)])
        b.wait()
        assert np.array_equal(by_place(b.hits(0)), want)
        assert np.array_equal(by_place(b.hits(2)), want)
        assert set(b.hits(1).tolist()) <= set(want[want["pos"] < 20].tolist())
        b.close()


def test_fetch_follows_keep():
    rng = np.random.default_rng(5)
    text, runs = stream(rng, 3000, 0.0)
    codes, _ = ba.pack(text)
    with scanner(rng, 0.3) as sc:
        room = np.empty(1, ba.HIT_DTYPE)
        assert sc.lib.blamm_hip_scan_fetch(sc.ctx, room.ctypes.data, 1) == ba.BLAMM_ERR_STATE
        n = ctypes.c_uint64()
        args = (sc.ctx, ba._ptr(codes, ctypes.c_uint64), None, 3000, ba._ptr(runs, ctypes.c_uint64), len(runs))
        assert sc.lib.blamm_hip_scan_keep(*args, ctypes.byref(n)) == 0 and n.value > 1
        assert sc.lib.blamm_hip_scan_fetch(sc.ctx, room.ctypes.data, 1) == ba.BLAMM_ERR_OVERFLOW
        room = np.empty(n.value, ba.HIT_DTYPE)
        assert sc.lib.blamm_hip_scan_fetch(sc.ctx, room.ctypes.data, n.value) == 0
        sc.reserve(1 << 20)
        assert sc.lib.blamm_hip_scan_fetch(sc.ctx, room.ctypes.data, n.value) == ba.BLAMM_ERR_STATE


def before_guard(a):
    """A copy of the words `a` (whole pages) that ends where a page which cannot
    be read begins."""
    m = mmap.mmap(-1, a.nbytes + mmap.PAGESIZE)
    room = np.frombuffer(m, np.uint64)
    at = room.ctypes.data
    room[:a.size] = a
    assert a.nbytes % mmap.PAGESIZE == 0
    libc = ctypes.CDLL(None, use_errno=True)
    assert libc.mprotect(ctypes.c_void_p(at + a.nbytes), ctypes.c_size_t(mmap.PAGESIZE), 0) == 0
    return room[:a.size]


@pytest.mark.parametrize("n", [1 << 15, 1 << 21])
def test_nothing_behind_the_last_base_is_read(n):
    """Host arrays of (n + 31) / 32 and (n + 63) / 64 words are enough for
    scans and histograms."""
    rng = np.random.default_rng(n)
    text, runs = stream(rng, n, 0.2)
    codes, lower = ba.pack(text)
    c, low = before_guard(codes[:n // 32]), before_guard(lower[:n // 64])
    with scanner(rng, 0.7) as sc:
        want = by_place(sc.scan(codes, n, runs, lower))
        assert len(want) > 100
        for scan in (sc.scan, sc.scan_pinned):
            assert np.array_equal(by_place(scan(c, n, runs, low)), want)
        ncols = 40
        lo, hi = np.full(ncols, -10, np.float32), np.full(ncols, 10, np.float32)
        assert np.array_equal(sc.hist(c, n, lo, hi, 50, runs, low), sc.hist(codes, n, lo, hi, 50, runs, lower))
