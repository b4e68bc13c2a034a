"""Where a recurrence's h lies in LDS (xcd_h_place and xcd_h_operand_piece in csrc/lstm_plan.h, compiled for the host): a permutation of the
16-byte pieces whose neighbours stay neighbours, of which the sparse operand takes every value once and every bank once per half
wavefront."""
import os
import shutil
import subprocess

import pytest

ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))

DRIVER = r"""
#include <cstdio>
#include "lstm_plan.h"
int main()
{
    for (int p = 0; p < 128; ++p) printf("%d\n", pimhip::xcd_h_place(p));
    for (int s = 0; s < 2; ++s)
        for (int lane = 0; lane < 64; ++lane) printf("%d\n", pimhip::xcd_h_operand_piece(s, lane));
}
"""


@pytest.fixture(scope="module")
def order(tmp_path_factory):
    """The place of every piece, and [register set][lane]: the first of the two neighbouring pieces that a lane reads half of."""
    if shutil.which("g++") is None:
        pytest.skip("no C++ compiler")
    d = tmp_path_factory.mktemp("lds_order")
    (d / "driver.cpp").write_text(DRIVER)
    subprocess.run(["g++", "-std=c++17", "-Wall", "-Werror", "-I", os.path.join(ROOT, "pimaicompiler_amd", "csrc"), str(d / "driver.cpp"), "-o",
                    str(d / "driver")], check=True, capture_output=True)
    lines = [int(line) for line in subprocess.run([str(d / "driver")], check=True, capture_output=True, text=True).stdout.split()]
    return lines[:128], [lines[128:192], lines[192:]]


def test_a_permutation_that_keeps_pairs(order):
    place = order[0]
    assert sorted(place) == list(range(128))
    assert all(place[p ^ 1] == place[p] ^ 1 and place[p] // 8 == p // 8 for p in range(128))


def test_the_operand_takes_every_half_piece_once(order):
    halves = [(piece + upper, lane % 2) for lanes in order[1] for lane, piece in enumerate(lanes) for upper in (0, 1)]
    assert sorted(halves) == [(p, half) for p in range(128) for half in (0, 1)]


def test_every_half_wavefront_reads_every_bank_once(order):
    place, operand = order
    for lanes in operand:
        for upper in (0, 1):
            for half in (range(32), range(32, 64)):
                banks = []
                for lane in half:
                    at = 16 * (place[lanes[lane]] ^ upper) + 8 * (lane % 2)
                    banks += [at // 4 % 64, (at // 4 + 1) % 64]
                assert sorted(banks) == list(range(64))
