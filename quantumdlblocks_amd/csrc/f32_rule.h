// Which fp32 kernel takes a launch: the wave-split ones (born_f32.h) with four
// waves a block or one, or the staged ones (born_fwd.h, born_bwd.h,
// purified.h).  Plain C++: a host test includes it.
#pragma once

#include <stdint.h>

namespace qdl {

constexpr int kF32MaxD = 128;  // wider heads take the staged kernels
constexpr int kF32Rows = 32;   // stationary rows per wave-split workgroup

constexpr int64_t f32_blocks(int64_t BH, int64_t T) { return (T + kF32Rows - 1) / kF32Rows * BH; }

// Waves per block of a wave-split launch: four, unless the blocks are many for
// their length.  One wave per block does without the reduction and the idle
// waves of short blocks, but its launch ends with whole blocks.  Up to padded
// head dim 64, where a CU holds two blocks of four waves, the two cross between
// 128 and 205 blocks per tile of the mean block.  Above, where it holds one and
// nothing runs beside its start and its reduction, already near 60 per tile of
// the longest block, once the blocks give most SIMDs a wave (with documents,
// whose ranges a block screens with its own threads, all of them: purified B4
// H16 T512 D128 with a 384-key window and documents of 128, 1024 blocks, 435
// and 317 us).  Steps with one wave and with four: B16 H16 T512 D32 241 and
// 290 us, B8 H8 T1024 D64 513 and 446, B8 H16 T512 D96 dense 543 and 642, B1
// H4 T8192 D128 with a 256-key window and no causality 5721 and 3493.  At
// padded head dims 96 and 128, over 1040 launches with both sides measured,
// the one taken is within 0.9% of the better on average (2.2% with 160 blocks
// per mean tile alone).
inline int f32_waves(int64_t BH, int64_t T, int D, bool causal, int64_t window, bool documents) {
    const int64_t tiles = (T + kF32Rows - 1) / kF32Rows, blocks = f32_blocks(BH, T);
    int64_t mean = causal ? (tiles + 1) / 2 : tiles, longest = tiles;
    if (causal && window > 0 && window / kF32Rows + 1 < longest) longest = window / kF32Rows + 1;
    if (longest < mean) mean = longest;
    if (blocks >= 160 * mean) return 1;
    return D > 64 && blocks >= 60 * longest && blocks >= (documents ? 1100 : longest < tiles ? 600 : 900) ? 1 : 4;
}

// Launches up to D = 128 that the staged kernels keep: without causality and
// with at least 256 blocks of their 128 rows (512 with a window, whose blocks
// differ in length; none at T below 128), at padded head dim 128, and the Born forward at 96 too.
// There the chip is full with either, and the four waves of a staged block
// read one tile where a wave-split wave reads its own.  With documents only
// the purified backward (the Born forward does not screen their ranges; the
// others are the faster ones with short documents).  Staged and wave-split:
// purified B16 H16 T512 D128 dense backward 1213 and 1602 us, forward 301 and
// 360; Born B8 H16 T512 D128 dense backward 641 and 847, forward 171 and 222;
// Born B8 H16 T512 D96 dense backward 437 and 404, forward 118 and 139.
inline bool f32_staged(bool purified, bool backward, int64_t BH, int64_t T, int D, bool causal, int64_t window,
                       bool documents) {
    if (D > kF32MaxD) return true;
    if (causal || T < 128 || (T + 127) / 128 * BH < (window > 0 ? 512 : 256)) return false;
    if (documents) return purified && backward && D > 96;
    return D > (purified || backward ? 96 : 64);
}

}  // namespace qdl
