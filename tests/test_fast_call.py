"""The extension module behind the Python front end (csrc/pybind_fast.cpp), as far as it goes without a GPU: argument
counts, keywords, rejected calls, and plans that notice what they were made from has changed."""
import ctypes

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


class FakeLibrary:
    """The entry points as Python functions: pulp_nn_add and the chain record the addresses they get, the others do nothing."""

    def __init__(self):
        self.seen, self.error, self.on_add, self.batch = [], 0, None, None
        nothing = ctypes.CFUNCTYPE(None)(lambda: None)
        add = ctypes.CFUNCTYPE(None, *[ctypes.c_void_p] * 3, *[ctypes.c_uint16] * 6)(self._add)
        chain = ctypes.CFUNCTYPE(None, *[ctypes.c_void_p] * 2, *[ctypes.c_uint16] * 3, ctypes.c_uint, ctypes.POINTER(api.HipBlock))(self._chain)
        last_error = ctypes.CFUNCTYPE(ctypes.c_int)(lambda: self.error)
        set_batch = ctypes.CFUNCTYPE(None, ctypes.c_uint)(lambda n: setattr(self, "batch", n))
        self.keep = dict.fromkeys(api.FAST_NAMES, nothing)
        self.keep.update(pulp_nn_add=add, pulp_nn_hip_dw_pw_chain_hwc=chain, pulp_nn_hip_last_error=last_error, pulp_nn_hip_set_batch=set_batch)

    def _add(self, a, b, out, m1, m2, shift, h, w, ch):
        self.seen.append((a, b, out))
        if self.on_add:
            self.on_add(len(self.seen), a)

    def _chain(self, x, out, w, h, c, n, blocks):
        self.seen.append((x, out) + tuple(blocks[i].dw_wt for i in range(n)))

    def bound(self):
        nn = api.PulpNN.__new__(api.PulpNN)
        nn._bind(32, {n: ctypes.cast(f, ctypes.c_void_p).value for n, f in self.keep.items()})
        nn.check = True
        nn._raise = self._raise
        return nn

    def _raise(self):
        code, self.error = self.error, 0
        raise api.PulpNNError(code, "fake")


def test_runs_of_one_plan_do_not_share_addresses():
    """A second run that is made while the first one queues (from another thread, here from inside a call)."""
    lib = FakeLibrary()
    marker = object()
    block = (7, None, None, None, 0, 0, 0, 0, 8, None, None, None, 0, 0, 0, 0)
    calls = [("pulp_nn_add", (marker, 1, 2, 1, 1, 1, 1, 1, 1)), ("pulp_nn_add", (3, marker, 4, 1, 1, 1, 1, 1, 1)),
             ("pulp_nn_hip_dw_pw_chain_hwc", (marker, 5, 1, 1, 1, [block, block]))]
    plan = api._fast.Plan(lib.bound(), 6, calls, marker, [])
    lib.on_add = lambda n, a: plan.run(2000) if n == 1 else None
    assert plan.run(1000) is True
    inner = [(2000, 1, 2), (3, 2000, 4), (2000, 5, 7, 7)]
    assert lib.seen == [(1000, 1, 2)] + inner + [(3, 1000, 4), (1000, 5, 7, 7)]
    assert lib.batch == 6
