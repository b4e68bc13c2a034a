"""The per-XCD recurrence around the lines between v_dot2 and sparse matrix instructions (xcd_on_dot in csrc/api_lstm.hip: below 8
steps, 12 from 513 to 640 units, not from 65 to 256 units), and stacks that were on v_dot2 before: the checks and bounds of
test_lstm_products_gpu.py at these sizes."""
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
