"""The extension module behind the Python front end (csrc/pybind_fast.cpp), as far as it goes without a GPU: argument
counts, keywords, rejected calls, and plans that notice what they were made from has changed."""
import pytest
import torch

from pulp_nn_amd import api

pytestmark = pytest.mark.skipif(api._fast is None, reason="extension not built")


@pytest.fixture
def nn():
    return api.PulpNN(32)


def test_arguments_are_converted_like_ctypes_did(nn):
    with pytest.raises(api.PulpNNError) as e:       # all arguments reach the library, which rejects the null pointers
        nn.pulp_nn_add(None, None, None, 1, 1, 1, 1, 1, 1)
    assert e.value.code == 1
    with pytest.raises(api.PulpNNError):            # keywords and defaults
        nn.hwc_to_chw(None, None, dim_x=1, dim_y=1, ch=1, pad_bottom=2)
    with pytest.raises(TypeError):
        nn.hwc_to_chw(None, None, dim_x=1, dim_y=1, channels=1)
    with pytest.raises(TypeError):
        nn.pulp_nn_add(None, None, None, 1, 1, 1, 1, 1, "x" if False else [])
    with pytest.raises(AssertionError):
        nn.pulp_nn_maxpool(None, None, 1, 2, 3)
    with pytest.raises(ValueError):                 # host tensors are refused
        nn.pulp_nn_add(torch.zeros(4, dtype=torch.uint8), None, None, 1, 1, 1, 1, 1, 1)
    nn.check = False
    nn.pulp_nn_add(None, None, None, 1, 1, 1, 1, 1, 1)
    assert nn.last_error() == 1
    nn.clear_error()
    nn.set_batch(3)
    assert nn.get_batch() == 3
    nn.set_batch(1)


def test_plan_notices_changed_entries(nn):
    marker, table = object(), {"shift": 3}
    calls = [("pulp_nn_add", (marker, None, None, 1, 1, 1, 1, 1, 1))]
    plan = api._fast.Plan(nn, 1, calls, marker, [(table, ("shift", "mult"))])
    with pytest.raises(api.PulpNNError):            # it runs: the library sees the null pointers
        plan.run(0)
    table["shift"] = int("3")
    with pytest.raises(api.PulpNNError):
        plan.run(0)
    table["mult"] = 1                               # an entry that was absent
    assert plan.run(0) is False
    del table["mult"]
    table["shift"] = 4
    assert plan.run(0) is False
    with pytest.raises(ValueError):
        api._fast.Plan(nn, 1, [("pulp_nn_nothing", ())], marker, [])
