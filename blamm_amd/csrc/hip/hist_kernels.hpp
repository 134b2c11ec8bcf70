// Empirical score histograms (`blamm hist -e`) on the split-BF16 engine.
//
// The reference fills them with the scan's sgemm (Histogram::histThread,
// hist.cpp:93-138) and bins the FP32 score of every window that satisfies the
// run rule (Histogram::extractObsScore, hist.cpp:70-91) with
// ScoreHistogram::addObservation (motif.h:96-102):
//   bin = clamp(int((score - min) / width), 0, nbins - 1),
//   width = (max - min) / nbins (motif.h:58-66), all in float.
// The score binned here is the FP32 sum of the window's weights in position
// order (lowercase bases contribute nothing).
//
// hist_filter_kernel scores windows with hi+lo MFMA tiles (those of the scan's
// split-BF16 form) and decides a window's bin from its MFMA score a when that is safe:
// x = fma(a, 1/width, -min/width) approximates the bin coordinate of the FP32
// score to within a per-column margin m (from the split and summation error
// bounds and the rounding of every float step, computed on the host), so when
// fract(x) lies in [m, 1 - m] the FP32 score's coordinate lies in the same
// unit interval and the bin is trunc(x), clamped (in LDS form the same in
// fixed point, see hist_rows).  Counts go to a
// workgroup-private LDS histogram that is added to HBM once per work item.
// Windows near a bin edge (about 2m of them) are staged per wave in LDS and
// binned exactly by the same wave (FP32 left-to-right sum of the window's
// weights, the reference's float arithmetic), so no record leaves the chip.
#pragma once

#include "scan_kernels.hpp"

namespace blamm {

// Fixed-point bin coordinates (LDS variant): the coordinate of a score, one
// up (so that rounding below bin 0 stays positive), plus 2^kHistInt in FP32 has
// the bin in the upper kHistInt bits of the mantissa and the fraction in the
// kHistFrac bits below.
constexpr int kHistInt = 10;
constexpr int kHistFrac = 23 - kHistInt;
constexpr uint32_t kHistMaxBins = 512;     // per column in LDS

struct HistSlot {
    float iw, c;       // x = fma(score, iw, c)
    float hm;          // bin decided from x iff |fract(x) - 1/2| <= hm
    float fc;          // LDS variant: x = fma(score, iw, fc) is c's coordinate + 1 + margin
    uint32_t fthr;     // LDS variant: bin undecided iff fraction << (32 - kHistFrac) < fthr
    float mn, wd;      // histogram minimum and bin width, as the reference computes them
    uint32_t len;      // motif length; 0 = empty slot
};

struct HistArgs {
    const uint64_t* packed;
    const uint64_t* lcmask;        // MASK variants only
    const uint4* frag_hi;
    const uint4* frag_lo;
    const HistSlot* hs;
    const float* slot_w;           // [slot][kMaxLen][4] FP32 weights
    const uint64_t* run_starts;
    const uint32_t* groups;        // group_pack(blk0, nch, 1 or 2): one column block per item, 2 = clamp (LDS variant)
    unsigned long long* counts;    // [slot][nbins]
    unsigned long long* counters;  // kCntBand: windows binned exactly; kCntQueue: work item head
    uint32_t nbases, nruns, qend, nbins;
    uint32_t ntiles, chunk_tiles, ngroups, nitems;
    uint32_t queue;                // work-item counter of this launch: counters[kCntQueue + queue]
};

// A block's LDS histogram, [bin][column]: a lane adds to its column's bank
// whatever its bin.  (With [column][bin] a wave's 64 adds met in random banks:
// ~31 cycles per ds_add.)  A bin below and one above the range take what
// rounds past its ends and are added to the first and last at the end.
__host__ __device__ constexpr uint32_t hist_words(uint32_t nbins)
{
    return (nbins + 2) * kBf16Cols;
}

// Undecided windows staged per wave before exact binning (8 KiB per block
// next to up to 64 KiB of histograms).
constexpr int kHistStage = 128;

// ScoreHistogram::addObservation's bin (motif.h:96-102) of an FP32 score:
// float subtract and IEEE division, then int() as the reference's x86-64
// hosts execute it (truncation; NaN or out of range gives INT_MIN), clamped.
__device__ __forceinline__ uint32_t hist_bin_ref(float s, float mn, float wd, uint32_t nbins)
{
    const float v = (s - mn) / wd;
    int b = (v >= -2147483648.0f && v < 2147483648.0f) ? (int)v : (int)0x80000000u;
    b = max(b, 0);
    b = min(b, (int)nbins - 1);
    return (uint32_t)b;
}

// Exact bins of staged windows: FP32 left-to-right sum of the window's weights
// (lowercase bases skipped), the reference's binning, one count each.  The
// run rule was applied when the record (first window of the lane, slot, rows)
// was staged.  Each lane takes one of the stage's last `take` <= 64 records and
// bins its first window; records with windows left go back to the stage, so
// that all lanes of a pass are busy (one pass over all windows of 65 to 128
// records ran with 12% of its lanes and took half of the kernel's time, in
// gathered loads).  Returns the number of windows this lane binned.
template <bool LDS>
__device__ __forceinline__ uint32_t hist_exact_pass(const HistArgs& a, Stage& st, uint32_t* hl, uint32_t blk0,
                                                    uint32_t take, uint32_t lane)
{
    const bool on = lane < take;
    st.n -= take;
    uint4 cd = make_uint4(0u, 0u, 0u, 0u);
    if (on) cd = st.buf[st.n + lane];
    const uint32_t q = cd.x + (on ? 8 * ((uint32_t)__builtin_ctz(cd.z) >> 2) + ((uint32_t)__builtin_ctz(cd.z) & 3) : 0u);
    cd.z &= cd.z - 1u;
    if (on) {
        const uint32_t slot = cd.y;
        const HistSlot h = a.hs[slot];
        const float* w = a.slot_w + (size_t)slot * kMaxLen * 4;
        const uint64_t bits = load_bits64(a.packed, 2ull * q);
        const uint64_t bits2 = h.len > 32 ? load_bits64(a.packed, 2ull * q + 64) : 0ull;
        const uint64_t mbits = a.lcmask ? load_bits64(a.lcmask, q) : 0ull;
        float s = 0.f;
        // eight loads at a time so that they overlap (rows up to kMaxLen exist
        // for every slot)
        for (uint32_t p0 = 0; p0 < h.len; p0 += 8) {
            const uint32_t src = (uint32_t)(p0 < 32 ? bits >> (2 * p0) : bits2 >> (2 * (p0 - 32)));
            float x[8];
#pragma unroll
            for (uint32_t u = 0; u < 8; ++u) x[u] = w[4 * (p0 + u) + ((src >> (2 * u)) & 3u)];
#pragma unroll
            for (uint32_t u = 0; u < 8; ++u)
                if (p0 + u < h.len && !((mbits >> (p0 + u)) & 1)) s += x[u];
        }
        const uint32_t bin = hist_bin_ref(s, h.mn, h.wd, a.nbins);
        if (LDS) atomicAdd(&hl[(bin + 1) * kBf16Cols + slot - blk0 * kBf16Cols], 1u);
        else atomicAdd(&a.counts[(size_t)slot * a.nbins + bin], 1ull);
    }
    const uint64_t m = __ballot(on && cd.z != 0u);
    if (m) {
        const uint32_t rank = __builtin_amdgcn_mbcnt_hi((uint32_t)(m >> 32), __builtin_amdgcn_mbcnt_lo((uint32_t)m, 0u));
        if (on && cd.z) st.buf[st.n + rank] = cd;
        st.n += (uint32_t)__popcll(m);
    }
    return on ? 1u : 0u;
}

// Does the window at q of length len end at or before the first run start
// after q?  rnext is the first run start after the tile's first window and jr
// its index (nbases past the last run).
__device__ __forceinline__ bool hist_row_fits(const HistArgs& a, uint32_t q, uint32_t len, uint32_t jr,
                                              uint32_t rnext)
{
    uint32_t r = rnext;
    if (q >= rnext) {
        uint32_t k = jr + 1;
        while (k < a.nruns && (uint32_t)a.run_starts[k] <= q) ++k;
        r = k < a.nruns ? (uint32_t)a.run_starts[k] : a.nbases;
    }
    return q + len <= r;
}

// The lane's binning values.
struct HistLane {
    float iw, c, hm, fc;
    uint32_t fthr, len, slot, hoff;
};

// Bins of one finished tile block (16 windows per lane).  A window whose
// bin the MFMA score decides adds 1 to it; the others add 0 (no branch, one
// LDS atomic per window) and are returned as a row mask for exact binning.
// FAST: every window fits its run and starts before qend.
// LDS variant, per window: one fma puts the coordinate in fixed point, a shift
// and a compare decide, a select and an add keep the row, a field extract and
// an add make the address: 7 instructions and the atomic.  CLAMP: scores of
// the block may lie outside the histograms' ranges.
template <bool FAST, bool LDS, bool CLAMP>
__device__ __forceinline__ uint32_t hist_rows(const HistArgs& a, uint32_t* hl, const f32x16& acc, const HistLane& h,
                                              uint32_t qlane, uint32_t jr, uint32_t rnext)
{
    const uint32_t live = h.len != 0 ? 1u : 0u;
    uint32_t valid = FAST ? (live ? 0xFFFFu : 0u) : 0u;
    if (!FAST) {
#pragma unroll
        for (int r = 0; r < 16; ++r) {
            const uint32_t q = qlane + 8 * (r >> 2) + (r & 3);
            valid |= (live && q < a.qend && hist_row_fits(a, q, h.len, jr, rnext) ? 1u : 0u) << r;
        }
    }
    uint32_t decided = 0;
    if constexpr (LDS) {
        const float top = (float)a.nbins + 1.5f;
#pragma unroll
        for (int r = 15; r >= 0; --r) {
            float x;
            if (CLAMP) x = __builtin_amdgcn_fmed3f(__builtin_fmaf(acc[r], h.iw, h.fc), 0.5f, top) + (float)(1 << kHistInt);
            else x = __builtin_fmaf(acc[r], h.iw, h.fc);
            const uint32_t word = __float_as_uint(x);
            const uint32_t ok = (word << (32 - kHistFrac)) >= h.fthr ? 1u : 0u;
            // (asm: the compiler takes three instructions each for the row's
            // bit and for the address)
            asm("v_lshl_add_u32 %0, %0, 1, %1" : "+v"(decided) : "v"(ok));
            uint32_t bin;
            asm("v_bfe_u32 %0, %1, %2, %3" : "=v"(bin) : "v"(word), "n"(kHistFrac), "n"(kHistInt));
            atomicAdd(&hl[bin * kBf16Cols + h.hoff], FAST ? ok : ok & (valid >> r));
        }
    } else {
        const int last = (int)a.nbins - 1;
#pragma unroll
        for (int r = 0; r < 16; ++r) {
            // (coordinates are below 2^30; a score that is no number becomes
            // one, which the columns with such scores never decide: hm < 0)
            const float x = __builtin_amdgcn_fmed3f(__builtin_fmaf(acc[r], h.iw, h.c), -0x1p30f, 0x1p30f);
            const bool ok = __builtin_fabsf(__builtin_amdgcn_fractf(x) - 0.5f) <= h.hm;
            const uint32_t bin = (uint32_t)min(max((int)x, 0), last);
            if (ok && ((valid >> r) & 1u)) atomicAdd(&a.counts[(size_t)h.slot * a.nbins + bin], 1ull);
            decided |= (ok ? 1u : 0u) << r;
        }
    }
    return ~decided & valid;
}

// Tiles t0, t0 + 4, ... < t1 of column block blk0 (the wave's share of a work
// item).  hl: the workgroup's LDS histogram of the item's columns (LDS
// variant).
template <int NCH, bool MASK, bool LDS, bool CLAMP>
__device__ __forceinline__ uint32_t hist_range(const HistArgs& a, Stage& st, uint32_t* hl, uint32_t blk0,
                                               uint32_t t0, uint32_t t1, uint32_t lane)
{
    uint32_t exact = 0;
    bf16x8 bh[1][NCH], bl[1][NCH];
#pragma unroll
    for (int j = 0; j < NCH; ++j) {
        const size_t idx = ((size_t)blk0 * kMaxChunks + j) * 64 + lane;
        bh[0][j] = __builtin_bit_cast(bf16x8, a.frag_hi[idx]);
        bl[0][j] = __builtin_bit_cast(bf16x8, a.frag_lo[idx]);
    }
    HistLane hv;
    hv.slot = blk0 * kBf16Cols + (lane & 31);
    {
        const HistSlot h = a.hs[hv.slot];
        hv.iw = h.iw;
        hv.c = h.c;
        hv.hm = h.hm;
        hv.fc = CLAMP ? h.fc : h.fc + (float)(1 << kHistInt);
        hv.fthr = h.fthr;
        hv.len = h.len;
        hv.hoff = lane & 31;
    }
    const uint32_t off = (lane & 31) + 2 * (lane >> 5);   // first base of the lane's window, 0..33
    // pk[t]: dwords 2t + off/16 and the next, so the window of tile t starts
    // at bit sh < 32 of pk[t]
    const uint32_t sh = 2 * (off & 15);
    const u64_a4* __restrict__ pk = (const u64_a4*)((const uint32_t*)a.packed + (off >> 4));
    const uint32_t* __restrict__ mk = (const uint32_t*)a.lcmask + (off >> 5);

    // run cursor: first run start after the current tile's first window
    uint32_t jr, rnext;
    {
        const uint32_t q = t0 * kBf16Tile;
        uint32_t l = 0, h = a.nruns;
        while (l < h) {
            const uint32_t mid = (l + h) >> 1;
            if ((uint32_t)a.run_starts[mid] <= q) l = mid + 1; else h = mid;
        }
        jr = __builtin_amdgcn_readfirstlane(l);
        rnext = __builtin_amdgcn_readfirstlane(l < a.nruns ? (uint32_t)a.run_starts[l] : a.nbases);
    }
    for (uint32_t t = t0; t < t1; t += kWavesPerBlock) {
        const uint32_t q0 = t * kBf16Tile;
        const OneHotSrc bits = onehot_src<NCH>(pk[t], pk[t + 1], pk[t + 2], sh);
        const uint64_t mb = MASK ? window_mask<NCH>(mk[t], mk[t + 1], mk[t + 2], off & 31) : 0ull;
        f32x16 acc[1];
        bf16_mfma_tile<NCH, 1, MASK>(acc, bh, bl, bits, mb);
        while (rnext <= q0) {
            ++jr;
            rnext = __builtin_amdgcn_readfirstlane(jr < a.nruns ? (uint32_t)a.run_starts[jr] : a.nbases);
        }
        // every window of the tile fits its run for every length <= 4 NCH
        const bool fast = q0 + (kBf16Tile - 1) + 4 * NCH <= rnext && q0 + kBf16Tile <= a.qend;
        const f32x16& av = acc_read(acc[0]);
        const uint32_t qlane = q0 + 4 * (lane >> 5);
        const uint32_t defer = fast ? hist_rows<true, LDS, CLAMP>(a, hl, av, hv, qlane, jr, rnext)
                                    : hist_rows<false, LDS, CLAMP>(a, hl, av, hv, qlane, jr, rnext);
        const uint64_t m = __ballot(defer != 0u);
        if (m) {
            while (st.n > (uint32_t)(kHistStage - 64)) exact += hist_exact_pass<LDS>(a, st, hl, blk0, 64u, lane);
            const uint32_t rank = __builtin_amdgcn_mbcnt_hi((uint32_t)(m >> 32),
                                                           __builtin_amdgcn_mbcnt_lo((uint32_t)m, 0u));
            if (defer) st.buf[st.n + rank] = make_uint4(qlane, hv.slot, defer, 0u);
            st.n += (uint32_t)__popcll(m);
        }
    }
    while (st.n) exact += hist_exact_pass<LDS>(a, st, hl, blk0, min(st.n, 64u), lane);
    return exact;
}

// Persistent: each workgroup takes work items (chunk of chunk_tiles tiles,
// column block) from one queue; its four waves share the item's tiles and
// its LDS histogram.  Up to 128 VGPRs so that four waves per SIMD hide the
// latency of the per-window binning.
// 10 Mbp x 1,000 columns x 250 bins: 4.1 ms, bound by VALU issue (11.7
// instructions per 64 windows, 3.2 ms of it).  8.7 ms before the exact passes
// filled their lanes (gathered weight loads, 1.5e8 wave loads against 2e7 now)
// and with 22 instructions per 64 windows in floating point.
// Blocks of motifs longer than 32 positions (WIDE: up to 16 chunks of hi and
// lo fragments in registers) run in a launch of their own at two waves per
// SIMD.
template <bool MASK, bool LDS, bool WIDE>
__global__ __launch_bounds__(kThreads, WIDE ? 2 : 4) void hist_filter_kernel(HistArgs a)
{
    extern __shared__ uint32_t hist_lds[];
    __shared__ uint4 stage_lds[kWavesPerBlock][kHistStage];
    __shared__ uint32_t item_s;
    const uint32_t lane = threadIdx.x & 63, wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
    Stage st{stage_lds[wave], 0u};
    uint32_t exact = 0;
    for (;;) {
        if (threadIdx.x == 0) item_s = (uint32_t)atomicAdd(&a.counters[kCntQueue + a.queue], 1ull);
        __syncthreads();
        const uint32_t it = __builtin_amdgcn_readfirstlane(item_s);
        if (it >= a.nitems) break;
        const uint32_t k = it / a.ngroups, g = it - k * a.ngroups;
        const uint32_t gp = __builtin_amdgcn_readfirstlane(a.groups[g]);
        const uint32_t blk0 = gp & 0xFFFFFu, nch = (gp >> 20) & 63u, nb = gp >> 26;
        const uint32_t t0 = k * a.chunk_tiles, t1 = min(t0 + a.chunk_tiles, a.ntiles);
        const uint32_t used = hist_words(a.nbins);
        if (LDS)
            for (uint32_t i = threadIdx.x; i < used; i += kThreads) hist_lds[i] = 0u;
        __syncthreads();
#define BLAMM_H(N) \
    case N * 8 + 1: exact += hist_range<N, MASK, LDS, false>(a, st, hist_lds, blk0, t0 + wave, t1, lane); break; \
    case N * 8 + 2: if constexpr (LDS) exact += hist_range<N, MASK, LDS, true>(a, st, hist_lds, blk0, t0 + wave, t1, lane); break;
        if constexpr (WIDE) {
            switch (nch * 8 + nb) {
                BLAMM_H(9) BLAMM_H(10) BLAMM_H(11) BLAMM_H(12)
                BLAMM_H(13) BLAMM_H(14) BLAMM_H(15) BLAMM_H(16)
                default: break;
            }
        } else {
            switch (nch * 8 + nb) {
                BLAMM_H(1) BLAMM_H(2) BLAMM_H(3) BLAMM_H(4)
                BLAMM_H(5) BLAMM_H(6) BLAMM_H(7) BLAMM_H(8)
                default: break;
            }
        }
#undef BLAMM_H
        if (LDS) {
            __syncthreads();
            unsigned long long* dst = a.counts + (size_t)blk0 * kBf16Cols * a.nbins;
            for (uint32_t i = threadIdx.x; i < kBf16Cols * a.nbins; i += kThreads) {
                const uint32_t col = i / a.nbins, bin = i - col * a.nbins;
                const uint32_t* h = hist_lds + col;
                uint32_t v = h[(bin + 1) * kBf16Cols];
                if (bin == 0) v += h[0];
                if (bin == a.nbins - 1) v += h[(a.nbins + 1) * kBf16Cols];
                if (v) atomicAdd(&dst[i], (unsigned long long)v);
            }
        }
        // the next item's first barrier orders these reads before its zeroing
    }
    // windows binned exactly (for statistics): one atomic per wave
    exact = __reduce_add_sync(~0ull, exact);
    if (lane == 0 && exact) atomicAdd(&a.counters[kCntBand], (unsigned long long)exact);
}

}  // namespace blamm
