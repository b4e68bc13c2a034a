"""Which kind of products the per-XCD LSTM kernel takes (csrc/lstm_plan.h), compiled for the host: where the measured lines lie."""
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
    long long H, T, chained;
    while (scanf("%lld %lld %lld", &H, &T, &chained) == 3) printf("%d\n", (int)pimhip::xcd_on_dot(H, T, (int)chained));
}
"""


@pytest.fixture(scope="module")
def on_dot(tmp_path_factory):
    if shutil.which("g++") is None:
        pytest.skip("no C++ compiler")
    d = tmp_path_factory.mktemp("lstm_plan")
    (d / "driver.cpp").write_text(DRIVER)
    subprocess.run(["g++", "-std=c++17", "-Wall", "-Werror", "-I", os.path.join(ROOT, "pimaicompiler_amd", "csrc"), str(d / "driver.cpp"), "-o",
                    str(d / "driver")], check=True, capture_output=True)

    def run(H, T, chained=1):
        out = subprocess.run([str(d / "driver")], input=f"{H} {T} {chained}", check=True, capture_output=True, text=True).stdout
        return bool(int(out))
    return run


@pytest.mark.parametrize("chained", [1, 2])
def test_few_units_stay_on_dot_at_any_length(on_dot, chained):
    assert on_dot(8, 4000, chained) and on_dot(56, 4000, chained) and not on_dot(72, 24, chained)


@pytest.mark.parametrize("H,chained,first_sparse", [(64, 1, 24), (128, 1, 8), (136, 1, 0), (256, 1, 0), (264, 1, 7), (512, 1, 7), (520, 1, 11), (656, 1, 11), (664, 1, 7),
                                                    (1024, 1, 7), (64, 2, 0), (256, 2, 0), (264, 2, 4), (520, 2, 7), (656, 2, 7), (664, 2, 4), (1024, 2, 4), (24, 3, 0),
                                                    (640, 3, 3), (664, 3, 0), (8, 4, 0), (640, 4, 0)])
def test_short_sequences_are_on_dot(on_dot, H, chained, first_sparse):
    assert not on_dot(H, max(first_sparse, 2), chained) and not on_dot(H, 4000, chained)
    assert first_sparse == 0 or on_dot(H, first_sparse - 1, chained) and on_dot(H, 2, chained)
