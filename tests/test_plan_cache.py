"""The cache of LSTM plans behind aten_lstm1 / aten_lstm2 (ops._plan_for), with a stand-in for the plan itself: no GPU needed."""
import pytest
import torch


@pytest.fixture
def cache(monkeypatch):
    from pimaicompiler_amd import ops as O
    built = []

    class Plan:
        def __init__(self, params, has_biases, num_layers, bidirectional, max_seq_len):
            self.max_seq_len = max_seq_len
            built.append(self)
    monkeypatch.setattr(O, "LstmPlan", Plan)
    monkeypatch.setattr(O, "_plan_cache", type(O._plan_cache)())
    O.built = built
    yield O
    del O.built


def weights():
    return [torch.randn(32, 8).half(), torch.randn(32, 8).half(), torch.randn(32).half(), torch.randn(32).half()]


def plan_for(O, params):
    return O._plan_for(params, True, 1, False, 4)


def test_weights_at_a_moved_tensors_old_address_can_be_invalidated(cache):
    params = weights()
    old = params[0].data                                   # (stands for whatever lies at that address next)
    first = plan_for(cache, params)
    params[0].data = torch.randn(32, 8).half()             # what Module.half() / .to() do
    assert cache.invalidate_lstm_plans([old]) == 1
    assert plan_for(cache, [old] + params[1:]) is not first


def test_a_moved_tensor_finds_the_plans_built_from_it(cache):
    params = weights()
    first = plan_for(cache, params)
    params[0].data = torch.randn(32, 8).half()
    assert cache.invalidate_lstm_plans([params[0]]) == 1
    assert plan_for(cache, params) is not first and len(cache.built) == 2


def test_an_address_in_the_cache_stays_taken(cache):
    """A plan reads its weights where they lay: that memory must not be given to other tensors while the plan is handed out."""
    params = weights()
    address = params[0].data_ptr()
    plan_for(cache, params)
    params[0].data = torch.randn(32, 8).half()
    others = [torch.empty(32, 8, dtype=torch.float16) for _ in range(64)]
    assert all(t.data_ptr() != address for t in others)
    assert plan_for(cache, params) is plan_for(cache, params)
    assert len(cache.built) == 2                           # one for the weights that were moved to


def test_an_update_in_place_is_seen(cache):
    params = weights()
    first = plan_for(cache, params)
    assert plan_for(cache, params) is first
    params[2].mul_(2)
    assert plan_for(cache, params) is not first
    assert cache.invalidate_lstm_plans([weights()[0]]) == 0 and cache.invalidate_lstm_plans() == 1
