"""How I_X_W products are cut into slices (csrc/vm_plan.h), compiled for the host: what the exchange of partial sums relies on, over
sizes at and around the edges of the rule."""
import itertools
import os
import shutil
import subprocess

import pytest

ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))

DRIVER = r"""
#include <cstdio>
#include "vm_plan.h"
int main()
{
    long long K, N, lda, addr;
    int cus;
    while (scanf("%lld %lld %lld %lld %d", &K, &N, &lda, &addr, &cus) == 5) {
        // (the results' address is given in the upper half of the weight's)
        const pimhip::VmPlan p = pimhip::vm_plan(K, N, lda, (uintptr_t)(addr & 0xffff), (uintptr_t)(addr >> 16), cus);
        printf("%d %d %d %d %zu %d\n", p.lanes_per_row, p.col_blocks, p.slices, p.rows_per_slice, pimhip::vm_max_partials(cus), (int)p.needs_no_workspace);
    }
}
"""

SIZES = (8, 9, 63, 64, 65, 84, 127, 129, 512, 513, 1000, 1023, 2048, 2357, 4096, 4951, 8191, 16384, 30001, 32768, 65535, 200000)


@pytest.fixture(scope="module")
def plans(tmp_path_factory):
    if shutil.which("g++") is None:
        pytest.skip("no C++ compiler")
    d = tmp_path_factory.mktemp("vm_plan")
    (d / "driver.cpp").write_text(DRIVER)
    subprocess.run(["g++", "-std=c++17", "-Wall", "-Werror", "-I", os.path.join(ROOT, "pimaicompiler_amd", "csrc"), str(d / "driver.cpp"), "-o",
                    str(d / "driver")], check=True, capture_output=True)

    def run(cases):
        text = "\n".join(" ".join(map(str, c)) for c in cases)
        out = subprocess.run([str(d / "driver")], input=text, check=True, capture_output=True, text=True).stdout
        return [tuple(map(int, line.split())) for line in out.splitlines()]
    return run


def test_partial_sums_of_every_product_fit_a_workspace_of_one_size(plans):
    """A workspace never grows, so no recorded graph can be left with the address of a freed one."""
    cases = [(k, n, n, 0, cus) for k, n, cus in itertools.product((0, 1) + SIZES, SIZES, (32, 64, 256, 304))]
    sliced = 0
    for (k, n, _, _, cus), (lanes, blocks, slices, rows, words, _) in zip(cases, plans(cases)):
        assert blocks == -(-n // (8 * lanes)) and slices >= 1
        assert (slices - 1) * rows < max(k, 1) <= max(slices * rows, 1) or k == 0   # the slices cover K, none is empty
        assert (slices - 1) * n <= words, (k, n, cus)
        assert words <= 64 * 1024 or cus > 512                                       # the static scratch array holds them as well
        sliced += slices > 1
    assert sliced > 100


def test_slices_of_a_large_weight_with_few_columns(plans):
    """A weight past 16 MB is read by about a block per CU, or by as many as sqrt(K / 10) slices give."""
    got = plans([(16384, 1024, 1024, 0, 256), (12000, 1024, 1024, 0, 256), (16384, 520, 520, 0, 256), (4096, 4096, 4096, 0, 256), (12896, 84, 84, 0, 256)])
    assert [(g[0], g[2]) for g in got] == [(16, 32), (16, 32), (16, 40), (16, 8), (8, 17)]


def test_small_and_odd_products_need_no_workspace(plans):
    """Weights of at most 256 KB, and operands of no whole 16-byte pieces (sizes, pitch, either address, any destination)."""
    cases, want = [], []
    for k, n, pitch, weight, results in itertools.product((513, 1024, 4951), (8, 64, 128, 136, 1301, 2048), (0, 3, 8), (0, 2, 8, 64), (0, 2, 48)):
        cases.append((k, n, n + pitch, weight | results << 16, 256))
        want.append(k * n * 2 <= 256 * 1024 or n % 8 != 0 or (n + pitch) % 8 != 0 or weight % 16 != 0 or results % 16 != 0)
    got = plans(cases)
    assert [bool(g[5]) for g in got] == want
    # ... and are cut like any other product of their size, so that their sums do not depend on where the records are
    assert all(g[2:4] == h[2:4] for g, h in zip(got, plans([(k, n, n, 0, cus) for k, n, _, _, cus in cases])))
