"""The autotuner's cache and candidates (needs the GPU)."""
from __future__ import annotations

import numpy as np
import pytest

import blamm_amd as ba
from blamm_amd import synth
from helpers import library, stream_case

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("prec", [ba.PREC_BF16X2, ba.PREC_BF16X2_LO, ba.PREC_FP32])
def test_entries_of_other_kernels_are_not_used(prec, tmp_path):
    """A cache line without the key's version, as written for other kernels and
    other meanings of the settings, is timed again; the bf16 forms, whose scans
    do not depend on the padding, keep 4."""
    import torch
    text, runs, bg = stream_case(33, 300_000)
    pwms, thr = library(synth.motifs(40, 5, 30, 0.5, seed=33), bg, pvalue=1e-4)
    P, lengths, _ = ba.build_pattern_matrix(pwms)
    packed, _ = ba.pack(text)
    cache = str(tmp_path / "tune.txt")
    with ba.HipScanner(0) as sc:
        sc.set_library(P, lengths, thr, prec)
        buf = np.zeros(int(sc.lib.blamm_hip_packed_words(len(text))), np.uint64)
        buf[:len(packed)] = packed
        codes = torch.from_numpy(buf.view(np.int64)).cuda()
        starts = torch.from_numpy(np.asarray(runs, np.uint64).view(np.int64)).cuda()
        args = (codes, None, len(text), starts, len(runs), cache)
        t, _ = sc.autotune(*args)
        if prec != ba.PREC_FP32:
            assert t.kpad_positions == 4
        key = open(cache).read().split()[0]
        version, rest = key.split("/", 1)
        assert version.startswith("t") and rest.startswith("gfx950/")
        for other in (rest, "t1/" + rest):
            with open(cache, "w") as f:
                f.write(f"{other} 7 1 8 0.001\n")
            t, ms = sc.autotune(*args)
            assert t.chunk_tiles != 7 and ms != 0.001
            assert open(cache).read().split("\n")[1].split()[0] == key
        with open(cache, "w") as f:
            f.write(f"{key} 7 1 4 0.5\n")
        t, ms = sc.autotune(*args)
        assert (t.chunk_tiles, t.blocks_per_wave, t.kpad_positions) == (7, 1, 4) and ms == 0.5
