"""Which kernel makes an input projection (csrc/xproj_plan.h), compiled for the host: the rule goes by tiles per CU, on a part of any
number of CUs."""
import os
import shutil
import subprocess

import pytest

ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))

DRIVER = r"""
#include <cstdio>
#include "xproj_plan.h"
int main()
{
    long long T, N;
    int count, packed, cus;
    while (scanf("%lld %lld %d %d %d", &T, &N, &count, &packed, &cus) == 5)
        printf("%d\n", cus == 0 ? (int)pimhip::context_most_positions(count, T) : pimhip::xproj_tile_rows(T, N, count, packed != 0, cus));
}
"""


@pytest.fixture(scope="module")
def rule(tmp_path_factory):
    if shutil.which("g++") is None:
        pytest.skip("no C++ compiler")
    d = tmp_path_factory.mktemp("xproj_plan")
    (d / "driver.cpp").write_text(DRIVER)
    subprocess.run(["g++", "-std=c++17", "-Wall", "-Werror", "-I", os.path.join(ROOT, "pimaicompiler_amd", "csrc"), str(d / "driver.cpp"), "-o",
                    str(d / "driver")], check=True, capture_output=True)

    def run(cases):
        text = "\n".join(" ".join(map(str, c)) for c in cases)
        return list(map(int, subprocess.run([str(d / "driver")], input=text, check=True, capture_output=True, text=True).stdout.split()))
    return run


def test_on_256_cus(rule):
    assert rule([(200, 4096, 1, 0, 256), (200, 4096, 1, 1, 256), (341, 4096, 1, 1, 256), (800, 1024, 1, 0, 256), (800, 4096, 1, 0, 256), (2048, 4096, 1, 0, 256),
                 (50, 4096, 2, 0, 256), (200, 4096, 2, 1, 256), (0x7fffffff, 0x7fffffff, 2, 0, 256)]) == [2, 0, 2, 0, 4, 4, 0, 2, 0]


@pytest.mark.parametrize("packed", [0, 1])
def test_half_the_cus_take_the_tiles_at_half_the_work(rule, packed):
    """A layer of half the columns on half the CUs has the same tiles per CU and takes the same kernel."""
    Ts = list(range(8, 1500, 56))
    full = rule([(T, 4096, 1, packed, 256) for T in Ts])
    assert full == rule([(T, 2048, 1, packed, 128) for T in Ts]) == rule([(T, 1024, 1, packed, 64) for T in Ts])
    assert set(full) == {0, 2, 4}


def test_one_layers_context_columns_stay_with_the_projection_kernels_for_long_sentences(rule):
    """(No CUs: the rule for the context columns of `count` layers, T wide.)"""
    def most(layers, width):
        return rule([(width, 0, layers, 0, 0)])[0]
    # (256, 512 wide, one layer: slower from about 60 positions on; 704 and more from about 100)
    assert most(1, 256) < 58 and most(1, 512) < 64 and 64 <= most(1, 704) < 96 and most(1, 1024) < 96
    assert all(most(n, h) == 160 for n in (2, 3, 4) for h in (256, 512, 1024))
