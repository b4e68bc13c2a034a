"""Which kind of products the per-XCD LSTM kernel takes (csrc/lstm_plan.h), compiled for the host: where the measured lines lie."""
import pytest

import test_lstm_products_gpu as products
import test_lstm_products_lines_gpu as lines
from lstm_kinds import on_dot


@pytest.mark.parametrize("chained", [1, 2])
def test_few_units_stay_on_dot_at_any_length(chained):
    assert on_dot(8, 4000, chained) and on_dot(56, 4000, chained) and not on_dot(72, 24, chained)


@pytest.mark.parametrize("H,chained,first_sparse", [(64, 1, 24), (128, 1, 8), (136, 1, 0), (256, 1, 0), (264, 1, 7), (512, 1, 7), (520, 1, 11), (656, 1, 11), (664, 1, 7),
                                                    (1024, 1, 7), (64, 2, 0), (256, 2, 0), (264, 2, 4), (520, 2, 7), (656, 2, 7), (664, 2, 4), (1024, 2, 4), (24, 3, 0),
                                                    (640, 3, 3), (664, 3, 0), (8, 4, 0), (640, 4, 0)])
def test_short_sequences_are_on_dot(H, chained, first_sparse):
    assert not on_dot(H, max(first_sparse, 2), chained) and not on_dot(H, 4000, chained)
    assert first_sparse == 0 or on_dot(H, first_sparse - 1, chained) and on_dot(H, 2, chained)


def test_sizes_of_the_gpu_tests_lie_on_the_sides_their_names_say():
    assert not any(on_dot(H, T) for H, T in products.ONE_SPARSE) and all(on_dot(H, T) for H, T in products.ONE_DOT)
    assert not any(on_dot(H, T, layers) for H, T in products.STACK_SPARSE for layers in (2, 4))   # (sums around a layer: always sparse)
    for before, behind in lines.ONE_LINES:
        assert on_dot(*before) and not on_dot(*behind)
    for (layers, *before), (layers_behind, *behind) in lines.PIPELINE_LINES:
        assert on_dot(*before, layers) and not on_dot(*behind, layers_behind)
