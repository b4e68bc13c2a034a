"""How a decoder step's rows are read (csrc/decoder_plan.h), compiled for the host: plain loads as long as all that a step reads fits the
caches, whichever operand makes up most of it, and for one of the two where that one alone fits the L2s and both do not."""
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
    {
        const pimhip::DecPlain p = pimhip::dec_plain_loads((int)layers, H, x_w, (int)ctx_layers, streamed != 0, enc_len, vocab);
        printf("%d %d\n", (int)p.layers, (int)p.classifier);
    }
}
"""


@pytest.fixture(scope="module")
def plain(tmp_path_factory):
    if shutil.which("g++") is None:
        pytest.skip("no C++ compiler")
    d = tmp_path_factory.mktemp("decoder_plan")
    (d / "driver.cpp").write_text(DRIVER)
    subprocess.run(["g++", "-std=c++17", "-Wall", "-Werror", "-I", os.path.join(ROOT, "pimaicompiler_amd", "csrc"), str(d / "driver.cpp"), "-o",
                    str(d / "driver")], check=True, capture_output=True)

    def run(*case):
        out = subprocess.run([str(d / "driver")], input=" ".join(map(str, case)), check=True, capture_output=True, text=True).stdout
        return tuple(map(bool, map(int, out.split())))
    return run


@pytest.fixture(scope="module")
def stay(plain):
    def layers(*case):
        kept, classifier = plain(*case)
        assert classifier
        return kept
    return layers


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


@pytest.mark.parametrize("case,want", [
    ((1, 1024, 1024, 0, 0, 0, 12200), (True, True)), ((1, 1024, 1024, 0, 0, 0, 12400), (False, True)),     # 39.8 and 40.2 MB
    ((2, 1024, 1024, 1, 0, 12, 8000), (True, True)), ((2, 1024, 1024, 1, 0, 12, 12400), (False, True)),    # both nearly fit, the classifier does not
    ((1, 1024, 1024, 0, 0, 0, 16384), (False, True)), ((1, 1024, 1024, 0, 0, 0, 16392), (True, False)),    # the classifier fits, the layers do
    ((1, 1024, 1024, 0, 0, 0, 32768), (True, False)), ((1, 1024, 1024, 0, 0, 0, 32776), (True, True)),     # 80 MB
    ((2, 1024, 1032, 1, 0, 12, 20000), (True, True)),                                                      # neither
    ((3, 1024, 1024, 2, 0, 12, 0), (False, True)), ((4, 1024, 1024, 3, 0, 12, 0), (False, True)), ((4, 1024, 2048, 3, 0, 12, 0), (True, True)),
    ((4, 1024, 1024, 3, 0, 12, 8000), (False, True)), ((4, 1024, 1024, 3, 0, 12, 9000), (True, True)),
    ((1, 896, 896, 0, 0, 0, 30000), (True, True)), ((1, 904, 904, 0, 0, 0, 30000), (True, False))])
def test_what_turns_the_l2s_over_is_read_past_them(plain, case, want):
    assert plain(*case) == want
