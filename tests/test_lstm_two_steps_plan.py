"""Whose projection two steps' launches make (csrc/lstm_plan.h), compiled for the host: not where W_ih is large and the projection's own
kernel streams it, so that reading it twice costs more than a launch; and where the measured lines lie."""
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
    long long dirs, layers, H, in_w, cus;
    while (scanf("%lld %lld %lld %lld %lld", &dirs, &layers, &H, &in_w, &cus) == 5)
        printf("%d\n", (int)pimhip::lstm_two_steps_project((int)dirs, (int)layers, H, in_w, (int)cus));
}
"""


@pytest.fixture(scope="module")
def in_the_steps(tmp_path_factory):
    if shutil.which("g++") is None:
        pytest.skip("no C++ compiler")
    d = tmp_path_factory.mktemp("two_steps")
    (d / "driver.cpp").write_text(DRIVER)
    subprocess.run(["g++", "-std=c++17", "-Wall", "-Werror", "-I", os.path.join(ROOT, "pimaicompiler_amd", "csrc"), str(d / "driver.cpp"), "-o",
                    str(d / "driver")], check=True, capture_output=True)

    def run(dirs, layers, H, in_w):
        out = subprocess.run([str(d / "driver")], input=f"{dirs} {layers} {H} {in_w} 256", check=True, capture_output=True, text=True).stdout
        return bool(int(out))
    return run


@pytest.mark.parametrize("dirs,layers,H,in_w", [(2, 1, 2056, 2056), (2, 2, 2056, 4112), (2, 2, 2048, 4096), (1, 1, 4096, 4096), (2, 1, 4096, 4096), (2, 1, 3072, 3072), (1, 1, 3072, 6144),
                                                (2, 1, 1536, 6144), (1, 2, 1024, 1024), (1, 4, 64, 64)])
def test_slower_in_the_steps(in_the_steps, dirs, layers, H, in_w):
    assert not in_the_steps(dirs, layers, H, in_w)


@pytest.mark.parametrize("dirs,layers,H,in_w", [(1, 1, 8, 8), (1, 1, 1024, 2048), (1, 1, 1024, 16384), (1, 1, 256, 16384), (1, 1, 1704, 1024), (1, 1, 2056, 8192), (1, 1, 3072, 3072),
                                                (2, 1, 1024, 1024), (2, 2, 512, 1024), (2, 1, 1024, 8192), (2, 1, 2056, 256), (1, 1, 4096, 256)])
def test_faster_in_the_steps(in_the_steps, dirs, layers, H, in_w):
    assert in_the_steps(dirs, layers, H, in_w)


def test_lines(in_the_steps):
    assert in_the_steps(1, 1, 4096, 1024) and not in_the_steps(1, 1, 4096, 1032)          # 32 MB, the kernel of tiles
    assert in_the_steps(2, 1, 2016, 2056) and not in_the_steps(2, 1, 2024, 2056)          # 128 tiles of 128 gate rows: that kernel's first
    assert in_the_steps(1, 1, 3072, 4096) and not in_the_steps(1, 1, 3072, 4104)          # 96 MB
    assert in_the_steps(1, 1, 2552, 16384) and not in_the_steps(1, 1, 2560, 16384)        # from 10240 gate rows on
