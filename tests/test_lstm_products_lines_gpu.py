"""The per-XCD recurrence on both sides of every line between v_dot2 and sparse matrix instructions (xcd_on_dot in csrc/lstm_plan.h; where
the lines lie is asked for in test_lstm_plan.py), and stacks of few steps with and without residual sums: the checks and bounds of
test_lstm_products_gpu.py at these sizes."""
import pytest

import test_lstm_products_gpu as products

pytestmark = pytest.mark.gpu
# (hidden size, steps): the last on v_dot2, the first on sparse instructions
ONE_LINES = [((64, 23), (64, 24)), ((128, 7), (128, 8)), ((264, 6), (264, 7)), ((512, 6), (512, 7)), ((520, 10), (520, 11)), ((656, 10), (656, 11)),
             ((664, 6), (664, 7)), ((1024, 6), (1024, 7))]
# the same with the layers in front
PIPELINE_LINES = [((2, 56, 30), (2, 64, 30)), ((2, 264, 3), (2, 264, 4)), ((2, 520, 6), (2, 520, 7)), ((2, 656, 6), (2, 656, 7)), ((2, 1024, 3), (2, 1024, 4)),
                  ((3, 16, 30), (3, 24, 30)), ((3, 640, 2), (3, 640, 3))]


@pytest.mark.parametrize("bidir", [False, True])
@pytest.mark.parametrize("H,T", [size for line in ONE_LINES for size in line] + [(8, 40), (56, 24), (72, 7), (136, 2), (256, 7)])
def test_single_layers(ops, H, T, bidir):
    products.test_every_step_is_as_close_to_64_bits_as_its_sums_allow(ops, H, T, bidir)


@pytest.mark.parametrize("layers,H,T", [size for line in PIPELINE_LINES for size in line] + [(2, 8, 30), (4, 16, 5), (4, 640, 2)])
def test_pipelines(ops, layers, H, T):
    products.test_stacks_match_libtorch(ops, H, T, layers, None)


@pytest.mark.parametrize("layers,res", [(2, None), (3, 1)])
@pytest.mark.parametrize("H,T", [(8, 4), (64, 40), (128, 40), (136, 4), (640, 4), (1024, 3)])
def test_stacks(ops, H, T, layers, res):
    products.test_stacks_match_libtorch(ops, H, T, layers, res)


@pytest.mark.parametrize("H,layers,bidir,short,long", [(128, 1, False, 7, 8), (264, 1, True, 6, 7), (640, 1, False, 10, 11), (1024, 1, True, 6, 7), (1024, 2, False, 3, 4),
                                                       (640, 3, False, 2, 3)])
def test_both_kinds_in_turn(ops, H, layers, bidir, short, long):
    products.test_one_plan_runs_both_kinds_in_turn(ops, H, layers, bidir, short, long)
