"""The calls that programs built on this engine make, for timing them.

A case is a dict of plain values; prepare() makes what such a program holds
before the call (a resident library, a packed stream, a batch slot), run()
makes the call through the public entry points of `blamm_amd` and work() says
what the call cannot do without.

Sizes follow the repository's own workloads (blamm_amd/synth.py): the example
scan of 1 Mbp against 128 columns, chromosomes against 1,000 to 2,000 motifs on
both strands, serving requests of ~4 Mbp that each ask for a part of a
resident library, and `hist -e` on the first 10 Mbp of a genome.  Motifs are
100 Dirichlet counts per position, sequences have a GC content of 0.35-0.50
with CG depleted, and runs end at N gaps or at the next sequence.

The engine reports hits in no fixed order, so every program that merges,
writes or compares them sorts them; run() does that on the device and returns
all of them as (position, column, score).
"""
from __future__ import annotations

import math

import numpy as np
import torch

import blamm_amd as ba

NUM_BINS = 250          # `blamm hist` default
PRECISIONS = {"bf16x2": ba.PREC_BF16X2, "bf16x2lo": ba.PREC_BF16X2_LO, "fp32": ba.PREC_FP32}


def _case(call, bases, motifs, lmin, lmax, pvalue, run=50_000, lower=0.0, precision="bf16x2", requests=1):
    """call: "device" (stream and hits stay on the GPU), "host" (host buffers
    in and out), "batch" (several requests in one launch) or "hist"."""
    return {"call": call, "bases": bases, "motifs": motifs, "lmin": lmin, "lmax": lmax,
            "pvalue": pvalue, "run": run, "lower": lower, "precision": precision, "requests": requests}


def _scan(name, *args, **more):
    return dict(_case(*args, **more), name=name)


def listed():
    return [
        # one gene's upstream region against a handful of motifs, from a
        # script or a notebook: nothing but the cost of a call
        _scan("one_gene", "host", 5_000, 10, 6, 20, 1e-4, run=5_000),
        # the example command: four 250 kbp records, 64 motifs on both strands
        _scan("example_set", "device", 1_000_000, 64, 6, 20, 1e-4, run=25_000),
        # one batch of the serving loop: requests of many short sequences, each
        # with its own motif subset of a resident library of 2,000
        _scan("serving_batch", "batch", 15_300_019, 2000, 5, 30, 1e-5, run=1_600, requests=5),
        # the headline: one genome group against a whole motif collection
        _scan("genome_group", "device", 62_500_000, 2000, 5, 30, 1e-5),
        # a chromosome arm at the default p-value, where hits are plenty
        _scan("chromosome", "device", 33_333_333, 1000, 5, 30, 1e-4),
        # the same through the command line's call: a soft-masked chromosome
        # (half of it lowercase) in host memory, hits back in host memory
        _scan("soft_masked", "host", 24_000_007, 500, 6, 25, 1e-5, run=30_000, lower=0.5),
        # an explorative threshold on promoters: hits dominate
        _scan("permissive", "device", 9_999_991, 300, 6, 25, 1e-3, run=2_000),
        # composite and zinc-finger motifs, longer than one packed word
        _scan("long_motifs", "device", 16_000_003, 300, 24, 60, 1e-5),
        # the FP32 form, by choice of the caller
        _scan("fp32_form", "device", 6_000_011, 500, 5, 30, 1e-4, precision="fp32"),
        # the split-BF16 form with the lo products
        _scan("lo_form", "device", 16_000_003, 500, 5, 30, 1e-4, precision="bf16x2lo"),
        # `hist -e` with its defaults: the first 10 Mbp, forward motifs only
        _scan("hist_default", "hist", 10_000_000, 1000, 5, 30, 0.0),
        # `hist -e` of a small set of sequences, some of it lowercase
        _scan("hist_small", "hist", 400_003, 64, 6, 20, 0.0, run=3_000, lower=0.2),
    ]


def _log(rng, lo, hi):
    return int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))


def draw(rng):
    call = rng.choice(["device", "device", "device", "host", "batch", "hist"])
    precision = rng.choice(["bf16x2"] * 6 + ["bf16x2lo", "fp32"]) if call == "device" else "bf16x2"
    lmin, lmax = rng.choice([(5, 30), (6, 20), (6, 25), (24, 60)])
    lower = rng.choice([0.0, 0.0, 0.1, 0.5])
    run = _log(rng, 500, 100_000)
    bases = _log(rng, 2_000, 62_500_000) | 1
    if call == "hist":
        bases = min(bases, 10_000_000)
        motifs = min(_log(rng, 8, 1000), max(8, int(1e10 / bases)))
        return _case(call, bases, motifs, lmin, lmax, 0.0, run, lower)
    # no more columns than the largest listed case scans in that form and
    # length, and about 5 million hits at most (a million where they come back
    # to the host)
    pvalue = rng.choice([1e-3, 1e-4, 1e-4, 1e-5, 1e-5, 1e-6])
    if lower:       # masked bases score 0: of use only where thresholds are above it
        lmin, lmax, pvalue = min(lmin, 6), min(lmax, 25), min(pvalue, 1e-5)
    most = {"bf16x2": 2.4e11, "bf16x2lo": 2.4e11, "fp32": 6e9}[precision]
    if lmax > 30 or lower:
        most /= 3
    cells = min(most, 5e6 / (pvalue + 5e-5))
    if call != "device":
        cells = min(cells, 1e6 / (pvalue + 5e-5))
    bases = min(bases, int(cells / 16) | 1)
    motifs = max(8, min(_log(rng, 8, 2000), int(cells / bases / 2)))
    requests = rng.randint(1, 12) if call == "batch" else 1
    return _case(call, bases, motifs, lmin, lmax, pvalue, run, lower, precision, requests)


def _columns(case):
    return case["motifs"] * (1 if case["call"] == "hist" else 2)


def _room(case):
    """Hits that a program makes room for: several times what the p-value asks
    for, and as many as short motifs have anyway (thresholds come from binned
    histograms, and a whole word of 5 bases is found every 1,024 bases)."""
    return int(_rate(case) * case["bases"] * _columns(case)) + 4096


def _rate(case):
    return 4 * case["pvalue"] + 8e-5 * (1 + 40 / case["motifs"])


def work(case):
    n, cols, mean = case["bases"], _columns(case), (case["lmin"] + case["lmax"]) / 2
    if case["call"] == "batch":      # requests ask for half of the library on average
        cols /= 2
    out = 8 * NUM_BINS * cols if case["call"] == "hist" else 16 * n * cols * case["pvalue"]
    return {"bytes": n * (0.375 if case["lower"] else 0.25) + 16 * mean * cols + out, "flops": 8.0 * n * cols * mean}


# ---- inputs ------------------------------------------------------------------

def _motifs(case, rng):
    """Count matrices (L x 4) with lengths uniform in lmin..lmax."""
    lengths = rng.integers(case["lmin"], case["lmax"] + 1, size=case["motifs"])
    counts = np.rint(100.0 * rng.dirichlet(np.full(4, 0.4), size=int(lengths.sum()))).astype(np.uint64)
    return np.split(counts, np.cumsum(lengths)[:-1])


def _bases(n, gc, gen):
    """Base codes with CG at about a fifth of its expected rate."""
    u = torch.rand(n, generator=gen, device="cuda")
    s = (u >= (1 - gc) / 2).to(torch.uint8) + (u >= 0.5).to(torch.uint8) + (u >= (1 + gc) / 2).to(torch.uint8)
    cg = torch.zeros(n, dtype=torch.bool, device="cuda")
    cg[1:] = (s[:-1] == 1) & (s[1:] == 2)
    v = torch.rand(n, generator=gen, device="cuda")
    return torch.where(cg & (v < 0.8), torch.where(v < 0.4, 0, 3).to(torch.uint8), s)


def _pack(codes):
    """2-bit codes, 32 to a 64-bit word."""
    pad = torch.zeros(-codes.numel() % 32, dtype=torch.uint8, device="cuda")
    c = torch.cat([codes, pad]).view(-1, 32)
    words = torch.zeros(c.shape[0], dtype=torch.int64, device="cuda")
    for i in range(32):
        words |= c[:, i].to(torch.int64) << (2 * i)
    return words


def _pack_bits(bits):
    pad = torch.zeros(-bits.numel() % 64, dtype=torch.bool, device="cuda")
    c = torch.cat([bits, pad]).view(-1, 64)
    words = torch.zeros(c.shape[0], dtype=torch.int64, device="cuda")
    for i in range(64):
        words |= c[:, i].to(torch.int64) << i
    return words


def _run_starts(n, mean, rng):
    """Sorted run starts: lognormal sequence lengths with the given mean."""
    k = int(1.5 * n / mean) + 16
    lens = np.maximum(8, np.rint(rng.lognormal(math.log(mean) - 0.32, 0.8, size=k))).astype(np.int64)
    starts = np.concatenate([[0], np.cumsum(lens)])
    return starts[starts < n].astype(np.uint64)


def _lower(n, frac, rng):
    """Repeats: lowercase intervals of ~1 kbp that cover about `frac`."""
    if not frac:
        return None
    flips = np.zeros(n + 1, np.int32)
    k = max(1, int(n * -math.log(1 - frac) / 1000))
    at = rng.integers(0, n, size=k)
    np.add.at(flips, at, 1)
    np.add.at(flips, np.minimum(n, at + rng.integers(50, 1950, size=k)), -1)
    return torch.from_numpy(flips).to("cuda")[:n].cumsum(0) > 0


def _inputs(case, seed):
    """Everything the case is made of, from the seed alone."""
    rng = np.random.default_rng([seed, case["bases"], case["motifs"]])
    gen = torch.Generator("cuda").manual_seed(int(rng.integers(1 << 62)))
    gc = float(rng.uniform(0.35, 0.50))
    pfms = _motifs(case, rng)
    n, nreq = case["bases"], case["requests"]
    share = rng.uniform(0.5, 1.5, size=nreq)
    cuts = np.concatenate([[0], np.rint(np.cumsum(share) / share.sum() * n).astype(np.int64)])
    codes = _bases(n, gc, gen)
    lower = _lower(n, case["lower"], rng)
    bg = torch.bincount(codes.to(torch.int32), minlength=4).cpu().numpy().astype(np.uint64) + np.uint64(1)
    pwms, thr = [], []
    for pfm in pfms:
        fwd = ba.pwm(pfm, bg, 0.25, False)
        if case["call"] == "hist":
            pwms.append(fwd)
            continue
        pwms += [fwd, ba.pwm(np.ascontiguousarray(pfm[::-1, ::-1]), bg, 0.25, True)]
        thr += [ba.pvalue_threshold(fwd, bg, case["pvalue"])] * 2
    thr = np.asarray(thr, np.float32)
    P, lengths, _ = ba.build_pattern_matrix(pwms)
    streams = []
    for r in range(nreq):
        a, b = int(cuts[r]), int(cuts[r + 1])
        cols = np.arange(len(pwms))
        if case["call"] == "batch":
            k = int(rng.integers(min(10, case["motifs"]), case["motifs"] + 1))
            pick = np.sort(rng.choice(case["motifs"], size=k, replace=False))
            cols = np.sort(np.concatenate([2 * pick, 2 * pick + 1]))
        streams.append((codes[a:b], None if lower is None else lower[a:b], _run_starts(b - a, case["run"], rng), cols))
    return P, lengths, thr, pwms, streams


def prepare(case, seed):
    P, lengths, thr, pwms, streams = _inputs(case, seed)
    sc = ba.HipScanner(0)
    ncols = len(pwms)
    st = {"call": case["call"], "sc": sc, "ncols": ncols, "room": _room(case)}
    codes, lower, runs, _ = streams[0]
    n = st["n"] = codes.numel()
    if case["call"] == "hist":
        sc.set_library(P, lengths, np.zeros(ncols, np.float32), ba.PREC_BF16X2)
        st["min"] = np.array([ba.min_score(w) for w in pwms], np.float32)
        st["max"] = np.array([ba.max_score(w) for w in pwms], np.float32)
    else:
        sc.set_library(P, lengths, thr, PRECISIONS[case["precision"]])
    if case["call"] in ("device", "hist"):
        words = torch.zeros(int(sc.lib.blamm_hip_packed_words(n)), dtype=torch.int64, device="cuda")
        words[:(n + 31) // 32] = _pack(codes)
        mask = None
        if lower is not None:
            mask = torch.zeros(int(sc.lib.blamm_hip_mask_words(n)), dtype=torch.int64, device="cuda")
            mask[:(n + 63) // 64] = _pack_bits(lower)
        st.update(words=words, mask=mask, runs=torch.from_numpy(runs.view(np.int64)).to("cuda"))
        if case["call"] == "device":
            sc.reserve(st["room"])
            st["hits"] = torch.empty(2 * st["room"], dtype=torch.int64, device="cuda")
            st["stream"] = torch.cuda.Stream()
        torch.cuda.synchronize()
    elif case["call"] == "host":
        st.update(words=_pack(codes).cpu().numpy().view(np.uint64), runs=runs,
                  mask=None if lower is None else _pack_bits(lower).cpu().numpy().view(np.uint64))
        if n * ncols > 1_000_000_000:
            sc.reserve(st["room"])
    else:
        reqs, st["rooms"] = [], [_room(case) for _ in streams]
        for codes, lower, runs, cols in streams:
            t = np.full(ncols, np.inf, np.float32)
            t[cols] = thr[cols]
            reqs.append(ba.ScanRequest(_pack(codes).cpu().numpy().view(np.uint64), codes.numel(), runs,
                                       None if lower is None else _pack_bits(lower).cpu().numpy().view(np.uint64), t,
                                       int(_rate(case) * codes.numel() * len(cols)) + 1024))
        st["reqs"] = reqs
        st["batch"] = ba.Batch(sc, max_bases=case["bases"] + 4096, max_requests=len(reqs))
    return st


# ---- one pass ----------------------------------------------------------------

def _sorted(h, ncols, room):
    """Device hit records ((n, 2) int64) sorted by position, then column, in a
    table with room for `room` hits (the rest is -1, -1, 0)."""
    key, order = torch.sort(h[:, 0] * ncols + (h[:, 1] & 0xFFFFFFFF))
    n = min(room, key.numel())
    key, order = key[:n], order[:n]
    pos = torch.full((room,), -1, dtype=torch.int64, device="cuda")
    col = torch.full((room,), -1, dtype=torch.int32, device="cuda")
    score = torch.zeros(room, dtype=torch.float32, device="cuda")
    pos[:n] = torch.div(key, ncols, rounding_mode="floor")
    col[:n] = key % ncols
    score[:n] = (h[:, 1] >> 32).to(torch.int32).view(torch.float32)[order]
    return {"pos": pos, "col": col, "score": score}


def _sorted_host(hits, ncols, room):
    """The same for hits in host memory: sorted there when they are few."""
    if hits.size >= 8192:
        return _sorted(torch.from_numpy(hits.view(np.int64).reshape(-1, 2)).to("cuda"), ncols, room)
    hits = hits[np.lexsort((hits["col"], hits["pos"]))][:room]
    n = hits.size
    pos, col, score = np.full(room, -1, np.int64), np.full(room, -1, np.int32), np.zeros(room, np.float32)
    pos[:n], col[:n], score[:n] = hits["pos"], hits["col"], hits["score"]
    return {"pos": pos, "col": col, "score": score}


def run(st):
    sc, ncols = st["sc"], st["ncols"]
    if st["call"] == "hist":
        counts = sc.hist_device(st["words"], st["mask"], st["n"], st["runs"], st["runs"].numel(), st["min"], st["max"],
                                NUM_BINS)
        return counts.view(np.int64)
    if st["call"] == "device":
        with torch.cuda.stream(st["stream"]):
            while True:
                sc.scan_device(st["words"], st["mask"], st["n"], st["runs"], st["runs"].numel(), st["hits"],
                               st["hits"].numel() // 2, None, st["stream"].cuda_stream)
                try:
                    n = sc.scan_finish()
                    break
                except ba.BlammError as e:      # the engine grew its scratch, or more hits than room: scan again
                    if e.code != ba.BLAMM_ERR_OVERFLOW:
                        raise
                    if 2 * sc.stats().hits > st["hits"].numel():
                        st["hits"] = torch.empty(2 * sc.stats().hits, dtype=torch.int64, device="cuda")
            return _sorted(st["hits"][:2 * n].view(n, 2), ncols, st["room"])
    if st["call"] == "host":
        scan = sc.scan if st["n"] * ncols <= 1_000_000_000 else sc.scan_pinned
        return _sorted_host(scan(st["words"], st["n"], st["runs"], st["mask"]), ncols, st["room"])
    b = st["batch"]
    b.submit(st["reqs"])
    b.wait()
    return [_sorted_host(b.hits(i), ncols, r) for i, r in enumerate(st["rooms"])]


# ---- the same in 64 bits -----------------------------------------------------

def exact(case, seed):
    """Every window's score as a product in 64 bits, and the windows at or above
    their threshold.  Empirical histograms are whole numbers: none."""
    if case["call"] == "hist" or case["bases"] * _columns(case) > 3e11:
        return None
    P, lengths, thr, _, streams = _inputs(case, seed)
    found = [_exact_stream(P, lengths, thr, stream, _room(case)) for stream in streams]
    return found if case["call"] == "batch" else found[0]


def _exact_stream(P, lengths, thr, stream, room):
    codes, lower, runs, cols = stream
    n, lmax = codes.numel(), P.shape[1] // 4
    W = torch.from_numpy(np.ascontiguousarray(P[cols].T)).to("cuda", torch.float64)
    t = torch.from_numpy(thr[cols]).to("cuda", torch.float64)
    L = torch.from_numpy(lengths[cols].astype(np.int64)).to("cuda")
    ids = torch.from_numpy(cols).to("cuda")
    starts = torch.from_numpy(runs.view(np.int64)).to("cuda")
    ends = torch.cat([starts[starts > 0], torch.tensor([n], device="cuda")])
    step = max(1024, min(1 << 20, int(4e8 / len(cols))))
    keys, scores = [], []
    for a in range(0, n, step):
        m = min(step, n - a)
        hot = torch.zeros(m + lmax, 4, dtype=torch.float64, device="cuda")
        c = codes[a:a + m + lmax].to(torch.int64)
        on = torch.ones(c.numel(), dtype=torch.float64, device="cuda") if lower is None else \
            (~lower[a:a + m + lmax]).to(torch.float64)
        hot[:c.numel()].scatter_(1, c[:, None], on[:, None])
        S = hot.view(-1).as_strided((m, 4 * lmax), (4, 1)).contiguous() @ W
        at = torch.arange(a, a + m, device="cuda")
        left = ends[torch.searchsorted(ends, at, right=True).clamp(max=ends.numel() - 1)] - at
        q, k = torch.nonzero((S >= t) & (L <= left[:, None]), as_tuple=True)
        keys.append((q + a) * len(lengths) + ids[k])
        scores.append(S[q, k])
    order = torch.argsort(torch.cat(keys))[:room]
    out = torch.zeros(room, dtype=torch.float64, device="cuda")
    out[:order.numel()] = torch.cat(scores)[order]
    return {"pos": None, "col": None, "score": out}
