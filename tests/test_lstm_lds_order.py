"""Where a recurrence's h lies in LDS (xcd_h_place in csrc/lstm_xcd_kernels.h): a permutation of the 16-byte pieces whose neighbours stay
neighbours, and every read of the sparse operand takes from all 64 banks once per half wavefront."""
import os
import re

ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))


def place():
    src = open(os.path.join(ROOT, "pimaicompiler_amd", "csrc", "lstm_xcd_kernels.h")).read()
    body = re.search(r"int xcd_h_place\(int p\) \{ return (.*?); \}", src).group(1)
    assert re.fullmatch(r"[p0-9\s^|&()<>]+", body)
    return lambda p: eval(body, {"p": p})


def test_a_permutation_that_keeps_pairs():
    f = place()
    assert sorted(f(p) for p in range(128)) == list(range(128))
    assert all(f(p ^ 1) == f(p) ^ 1 and f(p) // 8 == p // 8 for p in range(128))


def test_every_half_wavefront_reads_every_bank_once():
    f = place()
    for s in (0, 1):
        for upper in (0, 1):
            for half in (range(32), range(32, 64)):
                banks = []
                for lane in half:
                    at = 16 * (f(8 * (8 * s + ((lane & 15) >> 1)) + 2 * (lane >> 4)) ^ upper) + 8 * (lane & 1)
                    banks += [at // 4 % 64, (at // 4 + 1) % 64]
                assert sorted(banks) == list(range(64))
