"""How a decoder step's rows are read (csrc/decoder_plan.h), compiled for the host: plain loads as long as all that a step reads fits the
caches, whichever operand makes up most of it."""
import os
import shutil
import subprocess

import pytest

ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))

DRIVER = r"""
#include <cstdio>
#include "decoder_plan.h"
int main()
{
    long long layers, H, x_w, ctx_layers, streamed, enc_len, vocab;
    while (scanf("%lld %lld %lld %lld %lld %lld %lld", &layers, &H, &x_w, &ctx_layers, &streamed, &enc_len, &vocab) == 7)
        printf("%d\n", (int)pimhip::dec_rows_stay((int)layers, H, x_w, (int)ctx_layers, streamed != 0, enc_len, vocab));
}
"""


@pytest.fixture(scope="module")
def stay(tmp_path_factory):
    if shutil.which("g++") is None:
        pytest.skip("no C++ compiler")
    d = tmp_path_factory.mktemp("decoder_plan")
    (d / "driver.cpp").write_text(DRIVER)
    subprocess.run(["g++", "-std=c++17", "-Wall", "-Werror", "-I", os.path.join(ROOT, "pimaicompiler_amd", "csrc"), str(d / "driver.cpp"), "-o",
                    str(d / "driver")], check=True, capture_output=True)

    def run(*case):
        out = subprocess.run([str(d / "driver")], input=" ".join(map(str, case)), check=True, capture_output=True, text=True).stdout
        return bool(int(out))
    return run


# (layers, hidden units, inputs, layers with context, whether its columns are streamed, encoder outputs, classifier rows)
def test_the_classifier_counts(stay):
    assert stay(4, 1024, 1024, 3, 0, 12, 32000) and stay(4, 1024, 1024, 3, 0, 12, 88000)
    assert not stay(4, 1024, 1024, 3, 0, 12, 92000)


def test_context_columns_that_are_streamed_count(stay):
    assert stay(4, 1024, 1024, 3, 0, 12, 84000) and not stay(4, 1024, 1024, 3, 1, 12, 84000)
    assert not stay(4, 1024, 1024, 4, 0, 3000, 32000)            # and the products with a long sentence that stand in for them


@pytest.mark.parametrize("vocab", [0, 8000])
def test_a_wide_first_layer_counts(stay, vocab):
    assert stay(1, 1024, 28672, 0, 0, 0, vocab) and not stay(1, 1024, 40960, 0, 0, 0, vocab)
    assert not stay(2, 1024, 268435448, 1, 0, 12, vocab)         # the widest that a plan takes


def test_small_steps_stay(stay):
    assert stay(1, 8, 8, 0, 0, 0, 0) and stay(4, 1024, 1024, 4, 1, 0, 0)
