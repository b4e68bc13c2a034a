"""The per-XCD recurrence around the lines between v_dot2 and sparse matrix instructions (xcd_on_dot in csrc/lstm_plan.h), single layers,
pipelines of layers and stacks with residual sums: the checks and bounds of test_lstm_products_gpu.py at these sizes."""
import pytest

import test_lstm_products_gpu as products

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("bidir", [False, True])
@pytest.mark.parametrize("H,T", [(64, 7), (64, 8), (72, 7), (256, 7), (264, 7), (264, 8), (512, 8), (520, 11), (520, 12), (640, 12), (648, 7), (648, 8),
                                 (1024, 7), (1024, 8)])
def test_single_layers(ops, H, T, bidir):
    products.test_every_step_is_as_close_to_64_bits_as_its_sums_allow(ops, H, T, bidir)


@pytest.mark.parametrize("layers,res", [(2, None), (3, 1)])
@pytest.mark.parametrize("H,T", [(8, 4), (64, 40), (128, 40), (136, 4), (640, 4), (1024, 3)])
def test_stacks(ops, H, T, layers, res):
    products.test_stacks_match_libtorch(ops, H, T, layers, res)


@pytest.mark.parametrize("H,layers,bidir,short,long", [(64, 1, False, 7, 8), (512, 1, True, 7, 8), (640, 1, False, 11, 12), (1024, 1, True, 7, 8)])
def test_both_kinds_in_turn(ops, H, layers, bidir, short, long):
    products.test_one_plan_runs_both_kinds_in_turn(ops, H, layers, bidir, short, long)


@pytest.mark.parametrize("bidir", [False, True])
@pytest.mark.parametrize("H,T", [(8, 40), (56, 24), (64, 23), (64, 24), (128, 7), (128, 8), (136, 2), (264, 6), (656, 10), (656, 11), (664, 6), (664, 7)])
def test_single_layers_at_the_lines(ops, H, T, bidir):
    products.test_every_step_is_as_close_to_64_bits_as_its_sums_allow(ops, H, T, bidir)


@pytest.mark.parametrize("layers,H,T", [(2, 8, 30), (2, 56, 30), (2, 64, 3), (2, 264, 3), (2, 264, 4), (2, 520, 6), (2, 520, 7), (2, 656, 6), (2, 664, 4), (2, 1024, 2),
                                        (3, 16, 30), (3, 24, 30), (3, 640, 2), (3, 640, 3), (4, 16, 5), (4, 640, 2)])
def test_pipelines_at_the_lines(ops, layers, H, T):
    products.test_stacks_match_libtorch(ops, H, T, layers, None)


@pytest.mark.parametrize("H,layers,short,long", [(640, 2, 6, 7), (1024, 2, 3, 4), (640, 3, 2, 3)])
def test_both_kinds_of_pipelines_in_turn(ops, H, layers, short, long):
    products.test_one_plan_runs_both_kinds_in_turn(ops, H, layers, False, short, long)
