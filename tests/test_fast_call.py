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


@pytest.mark.gpu
def test_plan_asks_for_addresses_at_each_run(nn):
    """A chain's buffer that has other storage than when the plan was made: the run uses the new one.  A tensor without an
    address: an exception, at the call, at the plan and at the run."""
    marker = object()
    a, b, x, y = (torch.full((64,), v, dtype=torch.uint8, device="cuda") for v in (3, 5, 10, 20))
    out = torch.zeros(64, dtype=torch.uint8, device="cuda")
    nn.use_torch_stream()
    plan = api._fast.Plan(nn, 1, [("pulp_nn_add", (marker, a, out, 1, 1, 0, 1, 1, 64))], marker, [])
    assert plan.run(x) is True
    assert (out.cpu() == 13).all()
    a.set_(b)
    assert plan.run(y) is True
    assert (out.cpu() == 25).all()
    none = torch.zeros(64, dtype=torch.uint8, device="cuda").to_sparse()
    for refused in (lambda: nn.pulp_nn_add(none, a, out, 1, 1, 0, 1, 1, 64), lambda: plan.run(none),
                    lambda: api._fast.Plan(nn, 1, [("pulp_nn_add", (marker, none, out, 1, 1, 0, 1, 1, 64))], marker, [])):
        with pytest.raises((RuntimeError, ValueError)):
            refused()
