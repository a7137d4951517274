// When a 16-bit launch takes the few-block kernels (born_split16.h) instead of
// the tuned ones.
//
// Both sides end with their longest block.  A tuned kernel's walks the block's
// 64-row tiles one after the other; a split block's waves take a quarter of
// its 32-row tiles each, but every wave reads its tiles alone, so a launch
// also needs its tile bytes over what L2 delivers.  In microseconds,
//   tuned = ta + tc * (64-row tiles of the longest block)
//   split = sa + max(sc * (32-row tiles of the longest block) / 4, bytes / bw)
//           + 0.7 sa * (rounds of workgroups - 1)
// with the constants below, fitted per kernel and padded head dim to kernel
// times at B1 H4 T512 and T2048 (ta, tc, sa, sc: one workgroup per CU at most)
// and B2 H8 / B4 H12 T2048 (bw, GB/ms).  Tuned launches of several rounds take
// longer than this says, so the rule errs towards them; split is taken where
// it promises a tenth less (a quarter less with a window, whose blocks are
// mostly partly masked tiles).  Kernel times, tuned and split (causal, bf16):
//   B1 H4 T2048 D64    fwd 35.2 / 19.0   dQ 50.7 / 24.4   dK/dV 45.8 / 17.8
//   B2 H8 T2048 D64    fwd 35.9 / 22.2   dQ 53.3 / 30.6   dK/dV 48.6 / 33.6
//   B2 H16 T2048 D64   fwd 38.8 / 38.6   dQ 57.8 / 60.4   dK/dV 55.7 / 67.7
//   B4 H16 T1024 D64   fwd 22.2 / 26.3   dQ 34.1 / 42.2   dK/dV 31.1 / 44.8
//   B1 H4 T2048 D128   fwd 49.2 / 31.8   dQ 68.8 / 42.7   dK/dV 63.4 / 31.5
//   B2 H8 T2048 D128   fwd 51.8 / 54.3   dQ 75.9 / 75.0   dK/dV 69.0 / 82.7
// purified:
//   B2 H8 T2048 D64    fwd 70.2 / 33.0   dQ 73.6 / 41.0   dK/dV 72.5 / 45.8
//   B3 H6 T1100 D96    fwd 81.2 / 33.3   dQ 48.2 / 38.8   dK/dV 55.2 / 44.7 (fp16)
//   B4 H12 T2048 D128  fwd 99.6 / 172    dQ 107 / 207     dK/dV 188 / 273
#pragma once

#include <stdint.h>

namespace qdl {

enum SplitKernel : int { kSplitFwd = 0, kSplitDq = 1, kSplitDkdv = 2 };

struct SplitCost {
    double ta, tc, sa, sc, bw;
};

// [purified][padded head dim 32, 64, 96, 128, 256][kernel].
constexpr SplitCost kSplitCost[2][5][3] = {
    {{{5.6, 0.83, 5.9, 0.63, 8.8}, {4.8, 1.28, 7.3, 0.67, 5.4}, {3.5, 1.26, 3.8, 0.59, 7.2}},
     {{4.5, 0.94, 7.0, 0.83, 10.0}, {7.3, 1.35, 9.8, 0.94, 7.7}, {4.0, 1.30, 4.7, 0.89, 10.3}},
     {{3.2, 1.05, 8.2, 1.22, 6.0}, {7.7, 1.83, 10.6, 1.55, 4.6}, {5.4, 1.79, 5.6, 1.30, 6.5}},
     {{3.3, 1.43, 9.8, 1.43, 7.0}, {8.9, 1.92, 13.5, 1.90, 6.0}, {6.6, 1.78, 7.2, 1.45, 7.5}},
     {{4.0, 1.80, 6.0, 1.85, 9.8}, {6.0, 2.60, 9.0, 2.40, 6.9}, {8.0, 3.60, 8.0, 5.40, 3.1}}},
    {{{3.0, 1.98, 6.3, 1.14, 4.5}, {4.7, 1.99, 7.5, 1.03, 4.0}, {5.9, 1.95, 4.1, 0.98, 4.9}},
     {{4.0, 1.96, 7.6, 1.35, 6.1}, {6.9, 1.98, 10.6, 1.24, 5.2}, {5.3, 1.98, 5.3, 1.21, 7.2}},
     {{4.5, 2.33, 9.2, 1.81, 4.5}, {7.1, 2.20, 11.6, 1.86, 3.9}, {6.4, 2.55, 6.0, 1.66, 5.3}},
     {{4.8, 2.25, 11.0, 2.00, 5.2}, {10.2, 2.19, 14.6, 2.20, 4.3}, {7.3, 2.54, 7.3, 1.93, 6.1}},
     {{7.4, 2.60, 10.0, 2.00, 8.0}, {11.3, 2.55, 13.6, 2.20, 8.5}, {10.0, 5.00, 9.4, 5.95, 3.6}}}};

// Modelled times of one kernel and its rounds of workgroups; bh heads of T rows.
inline void split16_times(int kernel, bool pur, int64_t bh, int64_t T, int D, bool causal, int64_t window,
                          double* tuned, double* split, double* rounds) {
    const int d = D <= 128 ? (D + 31) / 32 - 1 : 4;
    const int dp = d < 4 ? 32 * (d + 1) : 256;
    const SplitCost& c = kSplitCost[pur ? 1 : 0][d][kernel];
    // Streamed rows a block of `rows` stationary ones spans, at most and in
    // the mean over the blocks.
    auto longest = [&](int64_t rows) {
        const int64_t n = (window > 0 && causal && window + rows < T) ? window + rows : T;
        return (double)n;
    };
    auto mean = [&](int64_t rows) {
        if (window > 0 && causal && window + rows < T) return (double)(window + rows);
        return causal ? 0.5 * (double)(T + rows) : (double)T;
    };
    const int64_t rows_tuned = kernel == kSplitDkdv || dp > 128 ? 128 : 256;
    const int64_t rows = kernel == kSplitDkdv || dp > 128 ? 32 : 64;
    const double blocks = (double)bh * (double)((T + rows - 1) / rows);
    const double bytes = blocks * mean(rows) / 32 * (128.0 * dp);  // two operands of 32 rows, 2 bytes
    const double chain = (double)(((int64_t)longest(rows) + 127) / 128);
    const double moved = bytes / (c.bw * 1e6);
    *tuned = c.ta + c.tc * (double)(((int64_t)longest(rows_tuned) + 63) / 64);
    const double slots = dp <= 64 ? 512 : 256;  // two workgroups per CU, or one (LDS)
    *rounds = (double)(int64_t)((blocks + slots - 1) / slots);
    *split = c.sa * (1.0 + 0.7 * (*rounds - 1)) + (c.sc * chain > moved ? c.sc * chain : moved);
}

// The kernels address a (T, D) slice with 32-bit byte offsets, rows up to T + 256.
constexpr bool split16_addressable(int64_t T) { return (T + 256) * 512 < ((int64_t)1 << 31); }

// Byte offset of a load within a slice: a chunk's offset in its tile (kSplitPastD
// for the chunks past D) and the tile's.  Unsigned, because the sum passes 2^31
// for chunks past D: it stays past the slice's end and below 2^32 for every
// addressable T (a signed sum overflows).
constexpr uint32_t kSplitPastD = 0x7ffffff0u;
constexpr uint32_t split16_load_at(uint32_t chunk, uint32_t tile) { return chunk + tile; }

// Rank of workgroup `bid` among a launch's blocks, longest tile ranges first.
// Where the whole launch is resident at once, two workgroups per CU (257 to
// 512 of them), the second half goes out shortest first, so that a CU pairs a
// long block with a short one (fp32 B2 H8 T1000 D64 step: 159 -> 142 us).
// Where only one fits, the second half starts as the first half's blocks end,
// and the longest of it must go first (causal, the pairing order and this one:
// fp32 B1 H8 T2048 D128 forward 121.6 and 99.2 us, backward 406 and 336;
// purified bf16 B1 H8 T4096 D128 forward 113.7 and 95.9; Born bf16 B1 H8 T2048
// D96 backward 76.4 and 70.3).
constexpr int split_rank(int bid, int grid, bool two_per_cu) {
    return two_per_cu && grid <= 512 && bid >= 256 ? grid - 1 - (bid - 256) : bid;
}
// Whether two workgroups of that much tile memory fit the 160 KiB of a CU
// (the rest of a workgroup's LDS is below 4 KiB).
constexpr bool split_two_per_cu(int tile_bytes) { return 2 * (tile_bytes + 4 * 1024) <= 160 * 1024; }

// bwd: dQ and dK/dV together (one side's row sums feed the other's kernel).
//
// The model takes a block's whole range for its length.  With document ids,
// whose lengths the host does not know, it may be a fraction of that, and then
// a split block's start weighs more than its chain.  At most head dims the
// split kernels stay ahead, or even, from documents of 128 tokens on.  Not so
// Born's at padded head dim 128, one block per CU with the longest start: the
// forward is no faster at a mean of 512 tokens and a fifth slower at 128, and
// the backward loses in launches of more than two rounds of blocks.  Tuned and
// split, by mean document length:
//   Born B1 H2 D128 dense        fwd T1000 512: 20.3 / 20.5   T1531 128: 19.2 / 24.0
//   Born B1 H8 T3000 D128        fwd 128: 19.5 / 35.7   bwd 128: 61.3 / 93.4
//   Born B1 H8 T1000 D96 dense   fwd 128: 17.9 / 20.7   bwd 128: 48.1 / 42.5
//   purified B2 H8 T1531 D96     fwd 128: 31.3 / 35.0   512: 66.9 / 40.6
template <class Args>
inline bool split16_pays(const Args& a, bool bwd, bool pur) {
    const int64_t bh = (int64_t)a.B * a.H;
    if (!split16_addressable(a.T)) return false;
    const bool born_docs = a.doc != nullptr && !pur && a.D > 96 && a.D <= 128;
    if (born_docs && !bwd) return false;
    double tuned = 0, split = 0;
    for (int k = bwd ? kSplitDq : kSplitFwd; k <= (bwd ? kSplitDkdv : kSplitFwd); ++k) {
        double t, s, rounds;
        split16_times(k, pur, bh, a.T, a.D, a.is_causal != 0, a.window, &t, &s, &rounds);
        if (born_docs && rounds > 2) return false;
        tuned += t;
        split += s;
    }
    return split < (a.window > 0 ? 0.75 : 0.9) * tuned;
}

}  // namespace qdl
