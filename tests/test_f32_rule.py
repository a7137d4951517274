"""Which fp32 kernel takes a launch (csrc/f32_rule.h), compiled on the host:
large launches without causality at padded head dims 96 and 128 keep the
staged kernels, and a block of the others gets one wave or four by the number
of blocks, each where it measured faster."""

from __future__ import annotations

import os
import shutil
import subprocess

import pytest

RULE = os.path.join(os.path.dirname(os.path.dirname(os.path.abspath(__file__))), "quantumdlblocks_amd", "csrc",
                    "f32_rule.h")
MAIN = """
#include <cstdio>
#include <cstdlib>
#include "%s"
int main(int, char** v) {
    const int64_t BH = atoll(v[1]), T = atoll(v[2]);
    const int D = atoi(v[3]), causal = atoi(v[4]), docs = atoi(v[6]);
    printf("%%d ", qdl::f32_waves(BH, T, D, causal, atoi(v[5]), docs));
    for (int pur = 0; pur < 2; ++pur)
        for (int bwd = 0; bwd < 2; ++bwd) printf("%%d ", qdl::f32_staged(pur, bwd, BH, T, D, causal, atoi(v[5]), docs));
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

    def ask(BH, T, D, causal=0, window=0, docs=0):
        """(waves per block, staged: Born forward, backward, purified forward, backward)"""
        args = [str(x) for x in (BH, T, D, causal, window, docs)]
        waves, *staged = subprocess.check_output([str(d / "rule"), *args], text=True).split()
        return int(waves), [w == "1" for w in staged]

    return ask


@pytest.mark.parametrize("BH,T,D,window,docs,staged", [
    (256, 512, 128, 0, 0, [1, 1, 1, 1]),   # full chips: both passes, Born and purified
    (32, 1000, 128, 0, 0, [1, 1, 1, 1]),
    (64, 1000, 104, 256, 0, [1, 1, 1, 1]),
    (128, 512, 96, 0, 0, [1, 0, 0, 0]),
    (128, 512, 72, 256, 0, [1, 0, 0, 0]),
    (128, 512, 128, 0, 1, [0, 0, 0, 1]),
    (128, 512, 96, 0, 1, [0, 0, 0, 0]),
    (128, 512, 64, 0, 0, [0, 0, 0, 0]),
    (255, 128, 128, 0, 0, [0, 0, 0, 0]),   # too few blocks of 128 rows
    (512, 100, 128, 0, 0, [0, 0, 0, 0]),   # none of them full
    (4, 8192, 128, 256, 0, [0, 0, 0, 0]),  # enough, but of unequal length
    (1, 64, 136, 0, 1, [1, 1, 1, 1]),      # wider heads: always
])
def test_staged_launches(rule, BH, T, D, window, docs, staged):
    assert rule(BH, T, D, 0, window, docs)[1] == [bool(x) for x in staged]
    assert rule(BH, T, D, 1, window, docs)[1] == [D > 128] * 4  # causal: never up to 128


# The faster side by more than a tenth, of launches measured with both.
@pytest.mark.parametrize("BH,T,D,causal,window,waves", [
    (128, 512, 128, 0, 0, 1), (8, 8192, 128, 1, 512, 1), (128, 512, 96, 0, 0, 1), (24, 1531, 128, 1, 512, 1),
    (64, 4096, 32, 1, 128, 1), (256, 512, 32, 1, 0, 1), (32, 512, 64, 1, 0, 4), (16, 1000, 64, 1, 0, 4),
    (4, 8192, 128, 0, 0, 4), (64, 384, 128, 1, 0, 4), (32, 700, 128, 1, 0, 4),
])
def test_waves_per_block(rule, BH, T, D, causal, window, waves):
    assert rule(BH, T, D, causal, window)[0] == waves


@pytest.mark.parametrize("BH,T,D,window,waves", [(64, 512, 128, 384, 4), (18, 1531, 96, 384, 4), (8, 8192, 96, 384, 1),
                                                 (128, 512, 96, 0, 1)])
def test_waves_per_block_with_documents(rule, BH, T, D, window, waves):
    assert rule(BH, T, D, 1, window, 1)[0] == waves
