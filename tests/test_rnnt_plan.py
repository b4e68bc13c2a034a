"""Which kernel the greedy decoding loop runs for a call (csrc/rnnt_plan.h), compiled for the host: a call of a few frames does not pay
for what only an utterance wins back, and the lines lie where they were measured."""
import os
import shutil
import subprocess

import pytest

ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))

DRIVER = r"""
#include <cstdio>
#include "rnnt_plan.h"
int main()
{
    long long vocab, joint, layers, frames;
    while (scanf("%lld %lld %lld %lld", &vocab, &joint, &layers, &frames) == 4)
        printf("%d %d\n", (int)pimhip::rnnt_greedy_every(vocab, layers, frames), pimhip::rnnt_greedy_own_rows(vocab, joint, layers, frames));
}
"""


@pytest.fixture(scope="module")
def kernel(tmp_path_factory):
    if shutil.which("g++") is None:
        pytest.skip("no C++ compiler")
    d = tmp_path_factory.mktemp("rnnt_plan")
    (d / "driver.cpp").write_text(DRIVER)
    subprocess.run(["g++", "-std=c++17", "-Wall", "-Werror", "-I", os.path.join(ROOT, "pimaicompiler_amd", "csrc"), str(d / "driver.cpp"), "-o",
                    str(d / "driver")], check=True, capture_output=True)

    def run(vocab, joint, layers, frames):
        out = subprocess.run([str(d / "driver")], input=f"{vocab} {joint} {layers} {frames}", check=True, capture_output=True, text=True).stdout
        every, rows = out.split()
        return bool(int(every)), int(rows)
    return run


@pytest.mark.parametrize("layers", [1, 2, 4])
@pytest.mark.parametrize("vocab", [1, 29, 32, 40, 64, 100, 128, 300, 512])
@pytest.mark.parametrize("frames", [0, 1, 4, 11])
def test_a_chunk_of_a_few_frames_starts_nothing_for_every_symbol(kernel, vocab, layers, frames):
    assert kernel(vocab, 512, layers, frames) == (False, 0)


@pytest.mark.parametrize("vocab,joint,layers,first,rows", [(1, 512, 1, 12, 0), (29, 512, 1, 15, 0), (64, 640, 1, 32, 0), (65, 640, 1, None, 0), (24, 512, 2, 12, 4),
                                                           (29, 512, 2, 15, 4), (32, 1024, 2, 16, 4), (32, 1032, 2, 16, 0), (33, 512, 2, 17, 8), (64, 512, 2, 32, 8),
                                                           (64, 520, 2, 32, 0), (100, 512, 3, 50, 0), (128, 512, 2, 64, 0), (129, 512, 2, None, 0)])
def test_the_line_lies_at_twelve_frames_and_half_the_symbols(kernel, vocab, joint, layers, first, rows):
    for frames in (12, 14, 15, 16, 17, 31, 32, 49, 50, 63, 64, 100, 1 << 31):
        every = first is not None and frames >= first
        assert kernel(vocab, joint, layers, frames) == (every, rows if every else 0)
