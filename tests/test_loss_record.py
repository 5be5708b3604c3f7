"""The loss records of a training step, whose values arrive when the step has been queued (CPU only)."""
import copy
import pickle
import types

import pytest


# (the package is imported when a test runs, not when it is collected: it loads the HIP runtime, and in a process that
# imports torch as well torch's has to come first)
def _metrics(count):
    from deepnet_amd.layer import _metrics
    return _metrics(count)


def Accumulate(stats, losses):
    from deepnet_amd.neuralnet import Accumulate
    return Accumulate(stats, losses)


def late(*args):
    from deepnet_amd.layer import late
    late(*args)


def settle(record):
    from deepnet_amd.layer import settle
    settle(record)


def _late(asked):
    perf = _metrics(10)

    def value():
        asked.append(1)
        return 2.5
    late(perf, 'error', value)
    return perf


@pytest.mark.parametrize("look", [lambda p: p.error, lambda p: vars(p)['error'], lambda p: p.__dict__['error'],
                                  lambda p: getattr(p, 'error'), lambda p: copy.copy(p).error, lambda p: pickle.loads(pickle.dumps(p)).error,
                                  lambda p: Accumulate([], [p])[0].error, lambda p: Accumulate([_metrics(3)], [p])[0].error,
                                  lambda p: eval(repr(p), {'LossRecord': types.SimpleNamespace, 'namespace': types.SimpleNamespace}).error])
def test_whoever_looks_at_a_record_gets_the_value(look):
    asked = []
    perf = _late(asked)
    assert look(perf) == 2.5 and perf.error == 2.5 and len(asked) == 1
    assert vars(perf) == dict(count=10, cross_entropy=0.0, correct_preds=0.0, error=2.5)


def test_records_are_compared_by_the_values_on_their_way():
    same = _metrics(10)
    same.error = 2.5
    assert _late([]) == same and same == _late([]) and _late([]) == _late([])
    assert _late([]) != _metrics(10) and _metrics(10) != _late([])
    assert _late([]) == types.SimpleNamespace(**vars(same)) and types.SimpleNamespace(**vars(same)) == _late([])
    assert _late([]) != 3


def test_a_deleted_field_stays_deleted():
    perf = _late([])
    del perf.error
    settle(perf)
    assert not hasattr(perf, 'error')


def test_several_fields_may_be_on_their_way():
    perf = _late([])
    late(perf, 'cross_entropy', lambda: 1.5)
    assert (perf.cross_entropy, perf.error, perf.count) == (1.5, 2.5, 10)
    late(perf, 'error', lambda: 3.5)
    settle(perf)
    settle(perf)
    assert vars(perf) == dict(count=10, cross_entropy=1.5, correct_preds=0.0, error=3.5)


def test_an_assigned_field_keeps_what_was_assigned():
    perf = _late([])
    perf.error = 7.0
    settle(perf)
    assert perf.error == 7.0
    perf = _late([])
    perf.error *= 2
    assert perf.error == 5.0


def test_a_value_that_cannot_be_had_is_not_zero():
    perf = _metrics(10)

    def value():
        raise RuntimeError('lost')
    late(perf, 'error', value)
    for _ in range(2):
        with pytest.raises(RuntimeError):
            perf.error
