"""The rule that sends a 16-bit launch of few blocks to the wave-split kernels
(csrc/split16_rule.h), compiled on the host: it takes the shapes their GPU
tests use, leaves the tuned kernels' own ranges alone, and stays finite at the
ends of the argument range."""

from __future__ import annotations

import heapq
import os
import shutil
import subprocess

import pytest

RULE = os.path.join(os.path.dirname(os.path.dirname(os.path.abspath(__file__))), "quantumdlblocks_amd", "csrc",
                    "split16_rule.h")
MAIN = """
#include <cstdio>
#include <cstdlib>
#include "%s"
struct A { int B, H, T, D, is_causal, window; };
int main(int, char** v) {
    const A a = {atoi(v[1]), atoi(v[2]), atoi(v[3]), atoi(v[4]), atoi(v[5]), atoi(v[6])};
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

    def ask(B, H, T, D, causal=1, window=0):
        """(Born forward, Born backward, purified forward, purified backward)"""
        args = [str(x) for x in (B, H, T, D, causal, window)]
        return [w == "1" for w in subprocess.check_output([str(d / "rule"), *args], text=True).split()]

    return ask


@pytest.mark.parametrize("D", [24, 64, 72, 96, 120, 128, 160, 256])
@pytest.mark.parametrize("causal,window", [(1, 0), (0, 0), (0, 300)])
def test_few_blocks_take_the_split_kernels(rule, D, causal, window):
    assert any(rule(1, 2, 700, D, causal, window))
    if window == 0:
        assert all(rule(1, 2, 1000, D, causal, window))


@pytest.mark.parametrize("B,H,T,D", [(16, 16, 1024, 64), (16, 16, 2048, 64), (32, 4, 1024, 64), (16, 8, 2048, 128),
                                     (4, 16, 8192, 64), (16, 4, 2048, 256), (2, 4, 64, 32), (1, 1, 1, 64),
                                     (4096, 4096, 4, 64), (1, 1, 1 << 28, 256)])
def test_others_keep_the_tuned_kernels(rule, B, H, T, D):
    assert not any(rule(B, H, T, D))


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
