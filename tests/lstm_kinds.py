"""Which kind of products the per-XCD LSTM kernel takes for a size: csrc/lstm_plan.h, compiled for the host."""
import functools
import os
import shutil
import subprocess
import tempfile

import pytest

ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))

DRIVER = r"""
#include <cstdio>
#include <cstdlib>
#include "lstm_plan.h"
int main(int, char** v) { printf("%d\n", (int)pimhip::xcd_on_dot(atoll(v[1]), atoll(v[2]), atoi(v[3]))); }
"""


@functools.lru_cache(None)
def _driver():
    if shutil.which("g++") is None:
        pytest.skip("no C++ compiler")
    d = tempfile.TemporaryDirectory()
    src, exe = os.path.join(d.name, "driver.cpp"), os.path.join(d.name, "driver")
    with open(src, "w") as f:
        f.write(DRIVER)
    subprocess.run(["g++", "-std=c++17", "-Wall", "-Werror", "-I", os.path.join(ROOT, "pimaicompiler_amd", "csrc"), src, "-o", exe], check=True,
                   capture_output=True)
    return d, exe


@functools.lru_cache(None)
def on_dot(H, T, chained=1):
    """v_dot2 (True) or sparse matrix instructions; `chained`: layers that one launch runs as a pipeline."""
    return bool(int(subprocess.run([_driver()[1], str(H), str(T), str(chained)], check=True, capture_output=True, text=True).stdout))
