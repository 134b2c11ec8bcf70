// The screen: the filter of the default scan form, and the first stage of the
// split-BF16 form's, on FP6 x FP4 matrix-core tiles.
//
// A scan must find every window whose score clears its column's threshold;
// nearly all of the ~1e11 windows of a scan are far below it.  The screen
// rules those out with an upper bound of the score in exact arithmetic:
// column c's weights become small integers y (FP6 E2M3: multiples of 1/8, at
// most 7.5) with
//     alpha_c w_c[p][b] <= y_c[p][b] + s_c[p]      for every base b,
// so a window can reach the threshold t only if
//     sum_p y_c[p][base(q+p)] >= alpha_c t - sum_p s_c[p].
// The left side is one row of v_mfma_f32_32x32x64_f8f6f4 per 16 positions:
// the window's one-hot row in FP4 times the column's integers in FP6.  Every
// product is a multiple of 1/16 below 4 and at most 64 of a sum are nonzero,
// so the FP32 accumulators hold the sums exactly, in any order.  Windows that
// pass become filter records and finalize_kernel decides them from the FP32
// weights (FP64 near the threshold), as before; no score comes from the
// screen.
//
// Why FP6: it runs at four times the BF16 rate and one instruction covers 16
// positions instead of 4.  The integers lose little: at 62.5 Mbp x 4,000
// columns, p = 1e-5, the screen records 13.95M lanes for 13.07M hits, a filter
// on the weights' bf16 hi terms with its proven band 14.53M (soft-masked
// streams, set 1 of the layout below: 465k against 315k for 259k hits).
//
// What bounds it: instruction issue beside the matrix cores.  Per 32 x 32 tile
// block a wave issues one MFMA per 16 positions (32 cycles of matrix core, 16
// of the issue port), 9 VALU instructions for the threshold test, a share of
// the 5 per step that build the rows, and a few on average to record windows:
// at 62.5 Mbp x 4,000 columns (motifs of 5-30, p = 1e-5) 1.54 MFMAs and 13.2
// VALU instructions, matrix cores busy 65 % of the time and VALU issue 69 %, at
// the 1.8 GHz that the card holds under this load.  10.0 ms against 22.2 ms for
// the BF16 filter, 42 against 93 ns per SIMD and tile block.
#pragma once

#include "scan_kernels.hpp"

namespace blamm {

typedef int i32x4 __attribute__((ext_vector_type(4)));
typedef int i32x6 __attribute__((ext_vector_type(6)));
typedef int i32x8 __attribute__((ext_vector_type(8)));

constexpr int kScreenPos = 16;                        // positions per MFMA
constexpr int kScreenSteps = kMaxLen / kScreenPos;    // MFMAs of the longest column
constexpr int kScreenFrag = 3;                        // uint2 per lane and step (32 FP6 values)
constexpr size_t kScreenBlock = (size_t)kScreenSteps * 64 * kScreenFrag;   // uint2 per column block

// Column blocks one wave scores at once for blocks of `steps` MFMAs, per unit
// of the motif-tile setting (1 or 2): the operand of a tile is built once for
// all of them (5 VALU instructions per step), and their FP6 fragments
// (6 registers per block and step) leave room for four waves per SIMD.
__host__ __device__ constexpr int screen_blocks(int steps, int unit)
{
    return unit * (steps == 1 ? 4 : steps == 2 ? 2 : 1);
}

struct ScreenArgs {
    const uint64_t* packed;
    const uint64_t* lcmask;          // MASK variants only
    const uint2* frag;               // [block][step][lane][kScreenFrag]
    const float* thr;                // per slot: threshold
    const double2* bound;            // per slot: accumulator bound = thr * x - y
    const uint32_t* groups;          // group_pack(first block, steps, blocks)
    uint4* cand;
    unsigned long long* counters;
    uint64_t cand_cap;
    // LO variants: the library's split-BF16 fragments, bands and lengths, and
    // the library slot of a batch's slot (list form)
    const uint4* hi;                 // [block][chunk][lane]
    const uint4* lo;
    const double* band;
    const int* len;
    const uint32_t* slot_map;
    const unsigned long long* before;   // if set: run only if that filter's records had no room
};

// Smallest accumulator value a window that reaches threshold t can have,
// rounded down.  The margin covers the rounding of the product and the
// difference.
__device__ __forceinline__ float screen_threshold(float t, double2 b)
{
    if (!__builtin_isfinite(t)) return t;
    const double m = (double)t * b.x;
    const double d = m - b.y;
    return __double2float_rd(d - (__builtin_fabs(m) + __builtin_fabs(b.y)) * 0x1p-50);
}

__device__ __forceinline__ f32x16 screen_mfma(i32x4 a, i32x6 b, f32x16 c)
{
    // FP4 (E2M1) rows, FP6 (E2M3) columns; unscaled
    const i32x8 A = __builtin_shufflevector(a, a, 0, 1, 2, 3, -1, -1, -1, -1);
    const i32x8 B = __builtin_shufflevector(b, b, 0, 1, 2, 3, 4, 5, -1, -1);
    return __builtin_amdgcn_mfma_scale_f32_32x32x64_f8f6f4(A, B, c, 4, 2, 0, 0, 0, 0);
}

// Bits of 16 consecutive bases of a 1-bit stream, those of the even bases at
// the bottom of a nibble each.
__device__ __forceinline__ uint32_t spread_even(uint32_t m)
{
    uint32_t v = __builtin_amdgcn_perm(0u, m, 0x0C010C00u);      // bytes b0 0 b1 0
    v = (v | (v << 4)) & 0x0F0F0F0Fu;
    return (v | (v << 2)) & 0x33333333u;
}

// The lane's rows of the one-hot operand.  Lane l holds positions
// 16 s + l/32 + 2 i (i = 0..7) of window l%32 in step s: x has the codes of 16
// consecutive bases from position 16 s + l/32 on, so bits 4i and 4i+1 are the
// code of the i-th of them.  Dword k marks base k: nibble i is 1 (FP4 0.5)
// where the base is k, so a row of four dwords is a shift and four
// three-input operations.  A lowercase base is marked nowhere.
template <int KS, bool MASK>
struct ScreenRows {
    i32x4 a[KS];
    __device__ __forceinline__ void build(const uint64_t (&w)[3], const uint32_t (&m)[3], uint32_t sh, uint32_t msh)
    {
        const uint32_t d[6] = {(uint32_t)w[0], (uint32_t)(w[0] >> 32), (uint32_t)w[1], (uint32_t)(w[1] >> 32),
                               (uint32_t)w[2], (uint32_t)(w[2] >> 32)};
        uint32_t mb[2] = {0u, 0u};
        if (MASK) {
            mb[0] = funnel32(m[0], m[1], msh);
            if (KS > 2) mb[1] = funnel32(m[1], m[2], msh);
        }
#pragma unroll
        for (int s = 0; s < KS; ++s) {
            const uint32_t x = funnel32(d[s], d[s + 1], sh), y = x >> 1;
            uint32_t on = 0x11111111u;
            if (MASK) on &= ~spread_even(mb[s >> 1] >> (16 * (s & 1)));
            a[s][0] = (int)(~x & ~y & on);
            a[s][1] = (int)(x & ~y & on);
            a[s][2] = (int)(~x & y & on);
            a[s][3] = (int)(x & y & on);
        }
    }
};

// The lane's number, computed where it is used: values made from it ahead of
// the tile loops would take registers that the fragments need.
__device__ __forceinline__ uint32_t screen_lane()
{
    uint32_t ones = ~0u;
    asm volatile("" : "+s"(ones));
    return __builtin_amdgcn_mbcnt_hi(ones, __builtin_amdgcn_mbcnt_lo(ones, 0u));
}

// Filter records staged per wave (as Stage, with the slice's base uniform).
// 512 halve the reservations of 256 and still leave LDS for four workgroups
// per CU (10 Mbp x 600 columns at p = 1e-3, 6.7M records: 0.56 -> 0.53 ms).
constexpr int kScreenStage = 512;
struct ScreenStage {
    uint4* buf;
    uint32_t n;
};

__device__ __forceinline__ void screen_flush(const ScreenArgs& a, ScreenStage& st)
{
    if (st.n == 0) return;
    const uint32_t lane = screen_lane();
    unsigned long long base = 0;
    if (lane == 0) base = atomicAdd(&a.counters[kCntCand], (unsigned long long)st.n);
    base = __shfl(base, 0);
    for (uint32_t i = lane; i < st.n; i += 64) {
        const uint64_t at = (uint64_t)base + i;
        if (at < a.cand_cap) a.cand[at] = st.buf[i];
    }
    st.n = 0;
}

// Record the lanes of a tile block that hold a window at or above th: the
// rows' mask is gathered from the sign bits of the differences (in asm so
// that these take one register, not sixteen, and stay behind the branch).
__device__ __forceinline__ void screen_emit(const ScreenArgs& a, ScreenStage& st, const f32x16& acc, float th,
                                            bool pred, uint64_t m, uint32_t t, uint32_t blk)
{
    if (st.n > (uint32_t)(kScreenStage - 64)) screen_flush(a, st);
    uint32_t below = 0;
#pragma unroll
    for (int r = 15; r >= 0; --r) {
        float d;
        asm volatile("v_sub_f32 %1, %2, %3\n\tv_alignbit_b32 %0, %0, %1, 31"
                     : "+v"(below), "=&v"(d)
                     : "v"(acc[r]), "v"(th));
    }
    const uint32_t lane = screen_lane();
    const uint32_t rank = __builtin_amdgcn_mbcnt_hi((uint32_t)(m >> 32), __builtin_amdgcn_mbcnt_lo((uint32_t)m, 0u));
    if (pred)
        st.buf[st.n + rank] = make_uint4(t * kBf16Tile + 4 * (lane >> 5), blk * kBf16Cols + (lane & 31),
                                         ~below & 0xFFFFu, 0u);
    st.n += (uint32_t)__popcll(m);
}

// The split-BF16 form (LO): a tile block that the screen cannot rule out is
// scored with the hi and lo products of its columns (as in bf16_mfma_tile), and
// its windows at or above thr - band, the proven band of that score, become
// records.  The screen marks such blocks over kSplitTiles tiles, one bit each,
// and this goes through the marked tiles ts + bit of one column block with the
// block's fragments in registers: read again for each tile block they are more
// than the caches deliver.  One tile block in seven is marked at p = 1e-4:
// 16 Mbp x 1,000 columns take 1.27 ms (2.35 with the fragments read for each,
// 2.05 with hi products for every window and lo products for blocks that pass;
// where nearly all are marked, 10 Mbp x 600 long columns at p = 1e-3, as much
// as the latter: 2.98).
constexpr uint32_t kSplitTiles = 64;

template <int KS, bool MASK, bool LIST>
__device__ __forceinline__ void screen_split(const ScreenArgs& a, ScreenStage& st, uint32_t blk, uint32_t ts,
                                             uint64_t marked)
{
    const uint32_t lane = screen_lane(), slot = blk * kBf16Cols + (lane & 31);
    uint32_t lib = slot;
    if constexpr (LIST) {
        lib = a.slot_map[slot];
        if (lib == kNoSlot) lib = 0;       // its threshold is +inf
    }
    const float th = thr_minus(a.thr[slot], a.band[lib]);
    const size_t row = (size_t)(lib / kBf16Cols) * kMaxChunks * 64 + (lane & 32) + lib % kBf16Cols;
    // chunks of four positions: up to three at the end may be empty
    constexpr int kFull = 4 * KS - 3;
    const int len = a.len[lib];
    int nch = kFull;
#pragma unroll
    for (int j = 0; j < 3; ++j) nch += __ballot(len > 4 * (kFull + j)) != 0;
    bf16x8 hi[4 * KS], lo[4 * KS];
#pragma unroll
    for (int j = 0; j < 4 * KS; ++j) {
        hi[j] = __builtin_bit_cast(bf16x8, a.hi[row + (size_t)j * 64]);
        lo[j] = __builtin_bit_cast(bf16x8, a.lo[row + (size_t)j * 64]);
    }
    const uint32_t off = (lane & 31) + 2 * (lane >> 5);   // first base of the lane's window, 0..33
    const uint32_t sh = 2 * (off & 15), po = 4 * (off >> 4), mo = 4 * (off >> 5);
    constexpr int NW = KS == 1 ? 1 : KS < 4 ? 2 : 3, NM = KS > 2 ? 3 : 2;
    uint64_t w[3] = {0, 0, 0};
    uint32_t mw[3] = {0, 0, 0};
    auto load = [&](uint32_t t) __attribute__((always_inline)) {
        const char* pk = (const char*)(a.packed + t);
#pragma unroll
        for (int i = 0; i < NW; ++i) w[i] = *(const u64_a4*)(pk + 8 * i + po);
        if (MASK) {
            const char* mk = (const char*)((const uint32_t*)a.lcmask + t);
#pragma unroll
            for (int i = 0; i < NM; ++i) mw[i] = *(const uint32_t*)(mk + 4 * i + mo);
        }
    };
    uint32_t t = ts + (uint32_t)__builtin_ctzll(marked);
    load(t);
    for (;;) {
        const OneHotSrc bits = onehot_src<4 * KS>(w[0], w[1], w[2], sh);
        const uint64_t mb = MASK ? window_mask<4 * KS>(mw[0], mw[1], mw[2], off & 31) : 0ull;
        marked &= marked - 1;
        const uint32_t now = t;
        if (marked) {
            t = ts + (uint32_t)__builtin_ctzll(marked);
            load(t);
        }
        f32x16 acc = {0.f};
        auto chunk = [&](int j) __attribute__((always_inline)) {
            const bf16x8 A = onehot_chunk<MASK>(bits, mb, j);
            acc = __builtin_amdgcn_mfma_f32_32x32x16_bf16(A, hi[j], acc, 0, 0, 0);
            acc = __builtin_amdgcn_mfma_f32_32x32x16_bf16(A, lo[j], acc, 0, 0, 0);
        };
#pragma unroll
        for (int j = 0; j < kFull; ++j) chunk(j);
        if (nch > kFull) {
            chunk(kFull);
            if (nch > kFull + 1) {
                chunk(kFull + 1);
                if (nch > kFull + 2) chunk(kFull + 2);
            }
        }
        const f32x16& v = acc_read(acc);
        const bool pred = tile_max(v) >= th;
        const uint64_t m = __ballot(pred);
        if (m) screen_emit(a, st, v, th, pred, m, now, blk);
        if (!marked) break;
    }
}

// Test block blk of tile t (LO: bit `bit` of mark).
template <bool LO>
__device__ __forceinline__ void screen_check(const ScreenArgs& a, ScreenStage& st, const f32x16& acc, float th,
                                             uint32_t t, uint32_t blk, uint32_t bit, uint64_t& mark)
{
    const f32x16& v = acc_read(acc);
    const bool pred = tile_max(v) >= th;
    const uint64_t m = __ballot(pred);
    if (m) {
        if constexpr (LO) mark |= 1ull << bit;
        else screen_emit(a, st, v, th, pred, m, t, blk);
    }
}

// Tiles [t0, t1) of column blocks blk0 .. blk0+NB-1.  Two accumulators
// alternate over the tile blocks: block b + 1's products (or the next tile's
// first) are issued before block b is tested, so the wave's own tests run
// beside its products.  LO: mark[b] gets block b's tiles, from t0 on.
template <int KS, int NB, bool MASK, bool LO>
__device__ __forceinline__ void screen_range(const ScreenArgs& a, ScreenStage& st, uint32_t blk0, uint32_t t0,
                                             uint32_t t1, uint64_t (&mark)[NB])
{
    const uint32_t lane = screen_lane();
    i32x6 B[NB][KS];
    float th[NB];
#pragma unroll
    for (int b = 0; b < NB; ++b) {
#pragma unroll
        for (int s = 0; s < KS; ++s) {
            const uint2* f = a.frag + ((size_t)(blk0 + b) * kScreenSteps + s) * 64 * kScreenFrag + lane * kScreenFrag;
            const uint2 f0 = f[0], f1 = f[1], f2 = f[2];
            B[b][s] = (i32x6){(int)f0.x, (int)f0.y, (int)f1.x, (int)f1.y, (int)f2.x, (int)f2.y};
        }
        const uint32_t slot = (blk0 + b) * kBf16Cols + (lane & 31);
        th[b] = screen_threshold(a.thr[slot], a.bound[slot]);
    }
    const uint32_t off = (lane & 31) + (lane >> 5);      // first base of the lane's row, 0..32
    const uint32_t sh = 2 * (off & 15), msh = off & 31;
    // words of tile t's rows: NW 64-bit words from dword 2t + off/16 on, NM
    // mask dwords from t + off/32 on; a uniform base and the lane's byte offset
    constexpr int NW = KS == 1 ? 1 : KS < 4 ? 2 : 3;
    constexpr int NM = KS > 2 ? 3 : 2;
    const uint32_t po = 4 * (off >> 4), mo = 4 * (off >> 5);
    uint64_t w[3] = {0, 0, 0};
    uint32_t mw[3] = {0, 0, 0};
    auto load = [&](uint32_t t) __attribute__((always_inline)) {
        const char* pk = (const char*)(a.packed + t);
#pragma unroll
        for (int i = 0; i < NW; ++i) w[i] = *(const u64_a4*)(pk + 8 * i + po);
        if (MASK) {
            const char* mk = (const char*)((const uint32_t*)a.lcmask + t);
#pragma unroll
            for (int i = 0; i < NM; ++i) mw[i] = *(const uint32_t*)(mk + 4 * i + mo);
        }
    };
    ScreenRows<KS, MASK> rows;
    load(t0);
    rows.build(w, mw, sh, msh);
    load(t0 + 1);
    auto product = [&](int b) __attribute__((always_inline)) {
        f32x16 acc = {0.f};
#pragma unroll
        for (int s = 0; s < KS; ++s) acc = screen_mfma(rows.a[s], B[b][s], acc);
        return acc;
    };
    if constexpr (NB == 1) {
        for (uint32_t t = t0; t < t1; ++t) {
            const f32x16 acc = product(0);
            rows.build(w, mw, sh, msh);
            load(t + 2);
            screen_check<LO>(a, st, acc, th[0], t, blk0, t - t0, mark[0]);
        }
    } else {
        static_assert(NB % 2 == 0, "block pairs alternate between two accumulators");
        f32x16 acc[2];
        acc[0] = product(0);
        for (uint32_t t = t0; t < t1; ++t) {
#pragma unroll
            for (int b = 0; b < NB; ++b) {
                if (b == NB - 1) {
                    // the rows of tile t + 1 (past the last tile: padding
                    // words, not tested)
                    rows.build(w, mw, sh, msh);
                    load(t + 2);
                }
                acc[(b + 1) & 1] = product((b + 1) % NB);
                screen_check<LO>(a, st, acc[b & 1], th[b], t, blk0 + b, t - t0, mark[b]);
            }
        }
    }
}

template <int KS, int NB, bool MASK, bool LIST, bool LO>
__device__ __forceinline__ void screen_tiles(const ScreenArgs& a, ScreenStage& st, uint32_t blk0, uint32_t t0,
                                             uint32_t t1)
{
    if constexpr (LO) {
        for (uint32_t t = t0; t < t1; t += kSplitTiles) {
            uint64_t mark[NB] = {};
            screen_range<KS, NB, MASK, true>(a, st, blk0, t, min(t1, t + kSplitTiles), mark);
#pragma unroll 1
            for (int b = 0; b < NB; ++b) {
                uint64_t m = mark[0];
#pragma unroll
                for (int i = 1; i < NB; ++i)
                    if (b == i) m = mark[i];
                if (m) screen_split<KS, MASK, LIST>(a, st, blk0 + b, t, m);
            }
        }
    } else {
        uint64_t mark[NB];
        screen_range<KS, NB, MASK, false>(a, st, blk0, t0, t1, mark);
    }
}

template <bool MASK, bool LIST, bool LO>
__device__ __forceinline__ void screen_item(const ScreenArgs& a, ScreenStage& st, uint32_t grp, uint32_t t0,
                                            uint32_t t1)
{
    const uint32_t blk0 = grp & 0xFFFFFu, steps = (grp >> 20) & 63u, nb = grp >> 26;
    switch (steps * 16 + nb) {
#define BLAMM_SCREEN(S, N) case S * 16 + N: screen_tiles<S, N, MASK, LIST, LO>(a, st, blk0, t0, t1); break;
    BLAMM_SCREEN(1, 8) BLAMM_SCREEN(1, 4) BLAMM_SCREEN(1, 2) BLAMM_SCREEN(1, 1)
    BLAMM_SCREEN(2, 4) BLAMM_SCREEN(2, 2) BLAMM_SCREEN(2, 1)
    BLAMM_SCREEN(3, 2) BLAMM_SCREEN(3, 1)
    BLAMM_SCREEN(4, 2) BLAMM_SCREEN(4, 1)
#undef BLAMM_SCREEN
    default: break;
    }
}

// (the LO variants' second look at a tile block takes registers of its own:
// three waves per SIMD)
template <bool MASK, bool LIST, bool LO>
__global__ __launch_bounds__(kThreads, LO ? 3 : 4) void screen_kernel(ScreenArgs a, WorkQueue q, ListArgs l)
{
    if (LO && a.before && a.before[kCntCand] <= a.cand_cap) return;
    __shared__ uint4 stage_lds[kWavesPerBlock][kScreenStage];
    ScreenStage st{stage_lds[__builtin_amdgcn_readfirstlane(threadIdx.x >> 6)], 0u};
    for_each_item<LIST>(a.counters, a.groups, q, l, [&](uint32_t grp, uint32_t t0, uint32_t t1) __attribute__((always_inline)) {
        screen_item<MASK, LIST, LO>(a, st, grp, t0, t1);
    });
    last_records(a, st.buf, st.n);
}

// ---------------------------------------------------------------------------
// Screen layout of a library, on the device: one wave per column slot, one
// lane per position.  Two sets are made: set 0 for streams without a
// lowercase mask, set 1 for masked ones.
//
// Set 0 subtracts a shift from each position's scaled weights before they are
// rounded (the shifts add up in the bound), so alpha can spread the widest
// position over all of -7.5..7.5, and the shift of the other positions is
// free: of 17 shifts and two roundings the lane keeps the one with the
// smallest expected slack s + y - alpha w under the motif's own base
// frequencies (~2^w), which is where the slack costs candidates.  In set 1 a
// lowercase base adds 0 to both sides, which a shift would break: weights are
// scaled by their largest magnitude and s >= 0 covers the rounding.  s is then
// all slack where the base is lowercase, which counts as much as the uppercase
// bases' (rounding up has none): without that every lowercase window of a
// 24-60 position column passes up to some bits above 0 (1 Mbp x 300 columns
// half lowercase, p = 1e-7: 1.6 times the windows of the BF16 filter, 1.49 ms;
// 1.0 times, 0.88 ms with it), for more records where hits are few and cost
// nothing (5-30 positions, p = 1e-5: 1.5 for 1.24 times, 0.06 ms both).
// ---------------------------------------------------------------------------
struct ScreenLayoutArgs {
    const float* slot_w;      // [slot][kMaxLen][4]
    const int* slot_len;
    uint2* frag[2];
    double2* bound[2];
    uint32_t nslots;
};

#ifndef BLAMM_INSTANTIATE
constexpr double kFp6Max = 7.5;

// x to a multiple of the FP6 grid in -7.5..7.5, nearest or upward.
__device__ __forceinline__ double fp6_round(double x, bool up)
{
    const double c = fmin(fmax(x, -kFp6Max), kFp6Max);
    const double m = fabs(c);
    const double step = m < 2.0 ? 0.125 : m < 4.0 ? 0.25 : 0.5;
    const double r = (up ? ceil(c / step) : rint(c / step)) * step;
    return fmin(fmax(r, -kFp6Max), kFp6Max);
}

// E2M3 code of a grid value: u eighths are 1.m x 2^(e-1) with one to three
// exponent steps.
__device__ __forceinline__ uint32_t fp6_code(double y)
{
    const uint32_t u = (uint32_t)(fabs(y) * 8.0);
    const uint32_t c = u < 16 ? u : u < 32 ? 8 + u / 2 : 16 + u / 4;
    return c | (y < 0.0 ? 32u : 0u);
}

__device__ __forceinline__ double wave_max(double v)
{
    for (int d = 32; d > 0; d >>= 1) v = fmax(v, __shfl_xor(v, d));
    return v;
}

__device__ __forceinline__ double wave_sum(double v)
{
    for (int d = 32; d > 0; d >>= 1) v += __shfl_xor(v, d);
    return v;
}

static __global__ __launch_bounds__(kThreads) void screen_layout_kernel(ScreenLayoutArgs a)
{
    constexpr int kDwords = kScreenSteps * 2 * 6;      // of a slot's fragments, per set
    __shared__ uint32_t frag[kWavesPerBlock][2][kDwords];
    const uint32_t lane = threadIdx.x & 63, wave = threadIdx.x >> 6;
    const uint32_t slot = blockIdx.x * kWavesPerBlock + wave;
    for (uint32_t i = lane; i < 2 * kDwords; i += 64) (&frag[wave][0][0])[i] = 0u;
    __syncthreads();
    // (an empty slot has zero weights and a +inf threshold)
    const int len = slot < a.nslots ? a.slot_len[slot] : 0;
    const bool in = (int)lane < len;
    double w[4], wmax = 0.0, wmin = 0.0, wabs = 0.0;
    float pi[4];
    for (int b = 0; b < 4; ++b) w[b] = in ? (double)a.slot_w[((size_t)slot * kMaxLen + lane) * 4 + b] : 0.0;
    wmax = fmax(fmax(w[0], w[1]), fmax(w[2], w[3]));
    wmin = fmin(fmin(w[0], w[1]), fmin(w[2], w[3]));
    wabs = fmax(fabs(wmax), fabs(wmin));
    for (int b = 0; b < 4; ++b) pi[b] = exp2f((float)fmax(w[b] - wmax, -60.0));
    const double half = wave_max((wmax - wmin) * 0.5), most = wave_max(wabs);
    // |FP64 left-to-right sum - exact sum| of any window
    const double fp64_err = wave_sum(wabs) * ((double)len * 0x1p-53 * (1.0 + 0x1p-20));
    for (int set = 0; set < 2; ++set) {
        const double range = set ? most : half;
        const double alpha = range > 0.0 ? kFp6Max / range : 1.0;
        double x[4], best_y[4] = {0.0, 0.0, 0.0, 0.0}, best_s = 0.0;
        for (int b = 0; b < 4; ++b) x[b] = alpha * w[b];
        const double xmax = alpha * wmax, xmid = 0.5 * (alpha * wmax + alpha * wmin);
        float best = 3.0e38f;
        for (int j = 0; j < (set ? 1 : 17); ++j) {
            // shifts around the middle of the position's range, then shifts
            // that bring its largest weight to 0..6
            const double o = j < 9 ? xmid + 0.25 * (j - 4) : xmax - (j == 9 ? 0.0 : j == 10 ? 0.5 : (double)(j - 10));
            const double off = set ? 0.0 : fmax(o, xmax - kFp6Max);
            for (int up = 0; up < 2; ++up) {
                double y[4], s = set ? 0.0 : -1e300;
                for (int b = 0; b < 4; ++b) {
                    y[b] = fp6_round(x[b] - off, up != 0);
                    s = fmax(s, x[b] - y[b]);
                }
                float slack = 0.f;
                for (int b = 0; b < 4; ++b) slack += pi[b] * (float)(s + y[b] - x[b]);
                if (set) slack += (pi[0] + pi[1] + pi[2] + pi[3]) * (float)s;
                if (slack < best) {
                    best = slack;
                    best_s = s;
                    for (int b = 0; b < 4; ++b) best_y[b] = y[b];
                }
            }
        }
        // rounding of x and of x - y
        const double s = in ? best_s + (alpha * wabs + 8.0) * 0x1p-50 : 0.0;
        const double sum = wave_sum(s), mag = wave_sum(fabs(s));
        if (in) {
            const uint32_t step = lane / kScreenPos, h = lane & 1, i = (lane % kScreenPos) >> 1;
            uint32_t* f = &frag[wave][set][(step * 2 + h) * 6];
            for (uint32_t b = 0; b < 4; ++b) {
                const uint32_t bit = 6 * (8 * b + i), c = fp6_code(best_y[b]);
                atomicOr(&f[bit / 32], c << (bit & 31));
                if ((bit & 31) > 26) atomicOr(&f[bit / 32 + 1], c >> (32 - (bit & 31)));
            }
        }
        if (lane == 0 && slot < a.nslots)
            // the operand's ones are FP4 0.5: half the sums
            a.bound[set][slot] = make_double2(0.5 * alpha, 0.5 * (alpha * fp64_err + sum + mag * 0x1p-46));
    }
    __syncthreads();
    if (slot >= a.nslots) return;
    for (uint32_t i = lane; i < 2 * kDwords; i += 64) {
        const uint32_t set = i / kDwords, d = i % kDwords, sh = d / 6;      // sh = step * 2 + half
        uint32_t* out = (uint32_t*)a.frag[set];
        const size_t row = ((size_t)(slot / kBf16Cols) * kScreenSteps + sh / 2) * 64 + (sh & 1) * 32 + slot % kBf16Cols;
        out[row * 6 + d % 6] = frag[wave][set][d];
    }
}
#endif

// Column blocks of a batch: batch slot s takes the screen fragments and bound
// of library slot slot_map[s] (an empty slot gets zeros; its threshold is
// +inf).
struct ScreenGatherArgs {
    const BatchDesc* desc;
    const uint32_t* slot_map;
    const uint2* lib_frag;
    const double2* lib_bound;
    uint2* out_frag;
    double2* out_bound;
};

#ifndef BLAMM_INSTANTIATE
static __global__ __launch_bounds__(256) void screen_gather_kernel(ScreenGatherArgs g)
{
    const uint32_t nblk = g.desc->nblk;
    const uint64_t stride = (uint64_t)gridDim.x * 256;
    const uint64_t t0 = (uint64_t)blockIdx.x * 256 + threadIdx.x;
    const uint64_t total = (uint64_t)nblk * kScreenBlock;
    for (uint64_t i = t0; i < total; i += stride) {
        const uint64_t row = i / kScreenFrag;
        const uint32_t l = (uint32_t)(row & 63), s = (uint32_t)((row >> 6) % kScreenSteps);
        const uint32_t b = (uint32_t)(row / (64 * kScreenSteps));
        const uint32_t lib = g.slot_map[b * kBf16Cols + (l & 31)];
        uint2 v = make_uint2(0u, 0u);
        if (lib != kNoSlot) {
            const size_t src = ((size_t)(lib / kBf16Cols) * kScreenSteps + s) * 64 + (l & 32) + lib % kBf16Cols;
            v = g.lib_frag[src * kScreenFrag + i % kScreenFrag];
        }
        g.out_frag[i] = v;
    }
    for (uint64_t s = t0; s < (uint64_t)nblk * kBf16Cols; s += stride) {
        const uint32_t lib = g.slot_map[s];
        g.out_bound[s] = lib != kNoSlot ? g.lib_bound[lib] : make_double2(0.0, 0.0);
    }
}
#endif

}  // namespace blamm
