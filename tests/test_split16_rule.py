"""The rule that sends a 16-bit launch of few blocks to the wave-split kernels
(csrc/split16_rule.h), compiled on the host: it takes each launch of their GPU
tests (test_gpu_split16.py, from the same lists), leaves the tuned kernels' own
ranges alone, and stays finite at the ends of the argument range."""

from __future__ import annotations

import heapq
import os
import shutil
import subprocess

import pytest

# name: (causal, window, documents)
MASKS = {
    "causal": (True, 0, False),
    "dense": (False, 0, False),
    "window": (True, 300, False),
    "window_nc": (False, 300, False),
    "docs": (True, 0, True),
    "docs_window": (True, 300, True),
    "docs_dense": (False, 0, True),
}
# What test_gpu_split16.py runs, as (B, H, T, D, mask).
HEAD_DIMS = [(1, 2, 1000, D, mask) for D in (24, 64, 72, 96, 120, 128, 160, 256) for mask in MASKS]
LENGTHS = [(1, 3, T, D, mask) for D, lengths in ((64, (449, 479, 480, 481, 512, 513, 1000)),
                                                 (128, (735, 736, 737, 767, 768, 833, 1000)))
           for T in lengths for mask in ("causal", "dense")]
WINDOW_NC_D128 = [(1, 2, 1500, D, "window_nc") for D in (120, 128)]
RAGGED_DOCS = [(B, 2, T, 64, mask) for B, T in ((1, 1301), (2, 705), (2, 1027)) for mask in ("docs", "docs_dense")]
UNSORTED_DOCS = [(2, 2, 600, 64, "docs")]
# 257 to 512 workgroups in some kernel: dK/dV (32-row blocks) or the forward and
# dQ (64-row ones), where two fit a CU (padded head dim 64) and where one does.
FULL_CHIP = [(1, 8, 1100, 64, "causal"), (2, 8, 1100, 64, "causal"), (2, 6, 1100, 96, "causal"),
             (1, 8, 1200, 128, "causal"), (1, 8, 1100, 160, "causal")]
FULL_CHIP_PURIFIED = [(2, 6, 1500, 96, "causal")]  # the Born forward of this one is a tuned kernel's

RULE = os.path.join(os.path.dirname(os.path.dirname(os.path.abspath(__file__))), "quantumdlblocks_amd", "csrc",
                    "split16_rule.h")
MAIN = """
#include <cstdio>
#include <cstdlib>
#include "%s"
struct A { int B, H, T, D, is_causal, window; const int* doc; };
int main(int, char** v) {
    const int id = 0;
    const A a = {atoi(v[1]), atoi(v[2]), atoi(v[3]), atoi(v[4]), atoi(v[5]), atoi(v[6]), atoi(v[7]) ? &id : nullptr};
    for (int pur = 0; pur < 2; ++pur)
        printf("%%d %%d ", qdl::split16_pays(a, false, pur), qdl::split16_pays(a, true, pur));
}
""" % RULE


@pytest.fixture(scope="module")
def rule(tmp_path_factory):
    gxx = shutil.which("g++")
    if gxx is None:
        pytest.skip("no host compiler")
    d = tmp_path_factory.mktemp("rule")
    (d / "main.cpp").write_text(MAIN)
    subprocess.run([gxx, "-std=c++17", str(d / "main.cpp"), "-o", str(d / "rule")], check=True)

    def ask(B, H, T, D, mask="causal"):
        """[Born forward, Born backward, purified forward, purified backward]"""
        args = [str(int(x)) for x in (B, H, T, D, *MASKS[mask])]
        return [w == "1" for w in subprocess.check_output([str(d / "rule"), *args], text=True).split()]

    return ask


@pytest.mark.parametrize("case", HEAD_DIMS, ids=str)
def test_every_head_dim_and_mask_takes_the_split_kernels(rule, case):
    """All four passes, but the Born forward at padded head dims 96 and 128
    with a window (too few tiles a block at this length) and at 128 with
    documents."""
    B, H, T, D, mask = case
    born_fwd = D <= 64 or D > 128 or mask in ("causal", "dense") or (D <= 96 and mask in ("docs", "docs_dense"))
    assert rule(*case) == [born_fwd, True, True, True]


@pytest.mark.parametrize("case", LENGTHS + WINDOW_NC_D128 + RAGGED_DOCS + UNSORTED_DOCS + FULL_CHIP, ids=str)
def test_launches_that_take_the_split_kernels_in_every_pass(rule, case):
    assert rule(*case) == [True] * 4


def test_full_chip_of_purified_blocks(rule):
    for case in FULL_CHIP_PURIFIED:
        assert rule(*case) == [False, True, True, True]


@pytest.mark.parametrize("B,H,T,D", [(16, 16, 1024, 64), (16, 16, 2048, 64), (32, 4, 1024, 64), (16, 8, 2048, 128),
                                     (4, 16, 8192, 64), (16, 4, 2048, 256), (2, 4, 64, 32), (1, 1, 1, 64),
                                     (4096, 4096, 4, 64), (1, 1, 1 << 28, 256)])
def test_others_keep_the_tuned_kernels(rule, B, H, T, D):
    assert not any(rule(B, H, T, D))


# Born launches with documents that measured faster on the tuned kernels.
@pytest.mark.parametrize("case,which", [((1, 8, 3000, 128, "docs"), 0), ((1, 8, 3000, 128, "docs"), 1),
                                        ((1, 2, 1531, 128, "docs_dense"), 0), ((1, 4, 3000, 120, "docs"), 0)])
def test_measured_slower_keep_the_tuned_kernels(rule, case, which):
    assert not rule(*case)[which]


OFFSETS = """
#include <initializer_list>
#include "%s"
using namespace qdl;
// In a constant expression an overflow of a signed sum is a compile error.
constexpr int64_t kMaxT = (((int64_t)1 << 31) - 1) / 512 - 256;
static_assert(split16_addressable(kMaxT) && !split16_addressable(kMaxT + 1), "the largest T");
constexpr bool past_the_slice(int64_t T) {
    for (int64_t D = 8; D <= 256; D += 8)
        for (int64_t row : {(int64_t)0, T / 2, T}) {  // a tile's first row; T: a tile that is not there
            const auto at = split16_load_at(kSplitPastD, (decltype(split16_load_at(0, 0)))(row * D * 2));
            if ((int64_t)(uint32_t)at < T * D * 2 || (int64_t)(uint32_t)at + 16 > ((int64_t)1 << 32)) return false;
        }
    return true;
}
static_assert(past_the_slice(1) && past_the_slice(32) && past_the_slice(1000) && past_the_slice(kMaxT), "chunks past D");
int main() {}
""" % RULE


def test_offsets_of_chunks_past_the_head_dim(tmp_path):
    """Loads of the columns past D stay out of a slice's range, without
    overflow, for every T that the kernels take."""
    gxx = shutil.which("g++")
    if gxx is None:
        pytest.skip("no host compiler")
    (tmp_path / "offsets.cpp").write_text(OFFSETS)
    subprocess.run([gxx, "-std=c++17", "-fsyntax-only", str(tmp_path / "offsets.cpp")], check=True)


ORDER = """
#include <cstdio>
#include <cstdlib>
#include "%s"
int main(int, char** v) {
    const int grid = atoi(v[1]);
    const bool two = qdl::split_two_per_cu(atoi(v[2]));
    printf("%%d ", two);
    for (int b = 0; b < grid; ++b) printf("%%d ", qdl::split_rank(b, grid, two));
}
""" % RULE


@pytest.mark.parametrize("tile_kib,per_cu", [(16, 2), (32, 2), (64, 2), (96, 1), (128, 1)])
def test_block_order_fits_the_workgroups_per_cu(tmp_path, tile_kib, per_cu):
    """Causal B1 H8 T2048 in 32-row blocks: 512 workgroups of 1 .. 64 tiles on
    256 CUs.  Where one fits a CU, each takes the next one as it ends, and an
    order that is not longest first ends later; where two fit, all start at
    once, the i-th and (i + 256)-th on one CU, and share its matrix pipes."""
    gxx = shutil.which("g++")
    if gxx is None:
        pytest.skip("no host compiler")
    (tmp_path / "order.cpp").write_text(ORDER)
    subprocess.run([gxx, "-std=c++17", str(tmp_path / "order.cpp"), "-o", str(tmp_path / "order")], check=True)
    got = subprocess.check_output([str(tmp_path / "order"), "512", str(tile_kib * 1024)], text=True).split()
    two, rank = got[0] == "1", [int(r) for r in got[1:]]
    assert two == (per_cu == 2) and sorted(rank) == list(range(512))
    tiles = [64 - r // 8 for r in rank]
    if two:
        end = max(tiles[i] + tiles[i + 256] for i in range(256))
    else:
        free = [0] * 256
        for t in tiles:
            heapq.heapreplace(free, free[0] + t)
        end = max(free)
    assert end <= 65
