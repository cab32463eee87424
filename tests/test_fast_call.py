"""The extension module behind the Python front end (csrc/pybind_fast.cpp), as far as it goes without a GPU: argument
counts, keywords, rejected calls, and plans that notice what they were made from has changed."""
import copy
import ctypes
import os
import subprocess
import sys
import types

import numpy as np
import pytest
import torch

from pulp_nn_amd import api, network

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
    marker, table = object(), {"shift": 100003}
    calls = [("pulp_nn_add", (marker, None, None, 1, 1, 1, 1, 1, 1))]
    plan = api._fast.Plan(nn, 1, calls, marker, [(table, ("shift", "mult"))])
    with pytest.raises(api.PulpNNError):            # it runs: the library sees the null pointers
        plan.run(0)
    equal = int("100003")
    assert equal is not table["shift"]              # an equal int that is another object: still what the plan was made from
    table["shift"] = equal
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


def test_a_library_object_without_init_raises():
    nn = api.PulpNN.__new__(api.PulpNN)
    for call in (lambda: nn.set_batch(1), lambda: nn.pulp_nn_add(None, None, None, 1, 1, 1, 1, 1, 1), lambda: api._fast.Plan(nn, 1, [], None, []),
                 lambda: api._fast.Plan.__new__(api._fast.Plan).run(None)):
        with pytest.raises(RuntimeError):
            call()


class TensorLike:
    """Has what the binding asks a tensor for."""
    is_cuda = True

    def __init__(self, address, contiguous=True):
        self.address, self.contiguous = address, contiguous

    def is_contiguous(self):
        return self.contiguous

    def data_ptr(self):
        return self.address


def test_arguments_that_were_taken_or_refused_still_are(nn):
    """What ctypes and the Python methods in front of it did: objects with a tensor's methods, error types, integers that
    have to be integers, an omitted scalar that is given as None."""
    lib = FakeLibrary()
    fake = lib.bound()
    fake.pulp_nn_add(TensorLike(0x1000), 0x2000, TensorLike(0x3000), 1, 1, 1, 1, 1, 1)
    assert lib.seen == [("pulp_nn_add", 0x1000, 0x2000, 0x3000)]
    host = TensorLike(0x1000)
    host.is_cuda = False
    for refused, error in ((TensorLike(0x1000, False), ValueError), (host, ValueError), ("text", AttributeError)):
        with pytest.raises(error):
            fake.pulp_nn_add(refused, None, None, 1, 1, 1, 1, 1, 1)
    fake.pulp_nn_add(0, 0, 0, 1.0, "1", True, np.int64(1), 1, 1)      # the reference's scalars: whatever int() takes
    for dim in (1.5, "1", None):                                     # the added entry points': integers
        with pytest.raises(TypeError):
            fake.hwc_to_chw(0, 0, dim, 1, 1)
        with pytest.raises(TypeError):
            fake.hwc_to_chw(0, 0, 1, 1, 1, pad_top=dim)
    fake.hwc_to_chw(0, 0, np.int32(1), 1, 1, pad_bottom=2)
    with pytest.raises(TypeError):                                   # counts: missing names, missing scalars
        fake.pulp_nn_linear(0, 0, 0, 0, 0, 0, 1, 1, 1, 1, 1)
    with pytest.raises(TypeError):
        fake.pulp_nn_maxpool(0)
    with pytest.raises(AssertionError):
        fake.pulp_nn_maxpool(0, 0, 1, 2, 3)
    for value in (1, "yes", 0, None):
        nn.check = value
        assert nn.check is bool(value)


POINTERS = dict({n: 7 for n in api.CONV_NAMES}, **{n: 8 for n in api.DW_NAMES}, pulp_nn_linear=6, pulp_nn_linear_out_32=4, pulp_nn_maxpool=2,
                pulp_nn_avgpool=2, pulp_nn_add=3, pulp_nn_depthwise_3x3_s1=2, pulp_nn_hip_hwc_to_chw=2, pulp_nn_hip_depthwise_hwc=6,
                pulp_nn_hip_dw_pw_hwc=2)


class FakeLibrary:
    """The entry points as Python functions that note the pointers they are given (their leading arguments)."""

    def __init__(self):
        self.seen, self.error, self.batch = [], 0, None
        self.on_call = lambda n, name, pointers: None   # n: how many calls there have been
        chain = ctypes.CFUNCTYPE(None, *[ctypes.c_void_p] * 2, *[ctypes.c_uint16] * 3, ctypes.c_uint, ctypes.POINTER(api.HipBlock))
        self.keep = {n: ctypes.CFUNCTYPE(None, *[ctypes.c_void_p] * k)(self._noter(n)) for n, k in POINTERS.items()}
        note = self._noter("pulp_nn_hip_dw_pw_chain_hwc")
        self.keep.update(
            pulp_nn_hip_dw_pw_chain_hwc=chain(lambda x, out, w, h, c, n, blocks: note(x, out, *(blocks[i].dw_wt for i in range(n)))),
            pulp_nn_hip_last_error=ctypes.CFUNCTYPE(ctypes.c_int)(lambda: self.error),
            pulp_nn_hip_clear_error=ctypes.CFUNCTYPE(None)(lambda: setattr(self, "error", 0)),
            pulp_nn_hip_set_batch=ctypes.CFUNCTYPE(None, ctypes.c_uint)(lambda n: setattr(self, "batch", n)))

    def _noter(self, name):
        def note(*pointers):
            self.error = 0
            self.seen.append((name,) + pointers)
            self.on_call(len(self.seen), name, pointers)
        return note

    def bound(self, cls=api.PulpNN):
        nn = cls.__new__(cls)
        nn._bind(32, {n: ctypes.cast(self.keep[n], ctypes.c_void_p).value for n in api.FAST_NAMES})
        nn.check, nn.bn_bits = True, 32
        nn._lib = types.SimpleNamespace(**self.keep, pulp_nn_hip_last_error_string=lambda: b"fake")
        return nn


def test_runs_of_one_plan_do_not_share_addresses():
    """A second run that is made while the first one queues (from another thread, here from inside a call)."""
    lib = FakeLibrary()
    marker = object()
    block = (7, None, None, None, 0, 0, 0, 0, 8, None, None, None, 0, 0, 0, 0)
    calls = [("pulp_nn_add", (marker, 1, 2, 1, 1, 1, 1, 1, 1)), ("pulp_nn_add", (3, marker, 4, 1, 1, 1, 1, 1, 1)),
             ("pulp_nn_hip_dw_pw_chain_hwc", (marker, 5, 1, 1, 1, [block, block]))]
    plan = api._fast.Plan(lib.bound(), 6, calls, marker, [])
    lib.on_call = lambda n, name, pointers: plan.run(2000) if n == 1 else None
    assert plan.run(1000) is True
    inner = [(2000, 1, 2), (3, 2000, 4), (2000, 5, 7, 7)]
    assert [c[1:] for c in lib.seen] == [(1000, 1, 2)] + inner + [(3, 1000, 4), (1000, 5, 7, 7)]
    assert lib.batch == 6


def test_plan_stops_at_a_call_without_a_kernel():
    """Code 2 is an answer, not an exception: the index of the call, for the caller to go on from."""
    lib = FakeLibrary()
    marker = object()
    plan = api._fast.Plan(lib.bound(), 1, [("pulp_nn_add", (marker, i, 2, 1, 1, 1, 1, 1, 1)) for i in range(3)], marker, [])

    def fail(code, when):
        def on_call(n, name, pointers):
            lib.error = code if when(n, *pointers) else 0
        lib.on_call = on_call

    fail(2, lambda n, a, b, out: b == 1 and a % 4)
    assert plan.run(1001) == 1 and len(lib.seen) == 2 and lib.error == 0
    lib.seen.clear()
    assert plan.run(1000) is True and len(lib.seen) == 3
    fail(1, lambda n, a, b, out: True)
    with pytest.raises(api.PulpNNError):
        plan.run(1000)


def bare_runner(nn, layers, input_shape, batch=1):
    """A runner whose tensors are addresses: the table's walk and its plan, without a GPU."""
    r = network.Runner.__new__(network.Runner)
    r.nn, r.layers, r.batch, r.fused, r.unfused = nn, layers, batch, True, set()
    r.fuse_blocks, r.unfused_blocks, r.launches, r.block_choice, r.chain_blocks, r.unchained = "auto", set(), 0, {}, True, set()
    r.shapes = network.infer_shapes(layers, input_shape)
    address = iter(range(0x10000, 0x7fffffff, 0x1000))
    r.params = [{k: next(address) for k in ("w", "bias", "k", "lam") if L.get(k) is not None} for L in layers]
    r.act = {L["name"]: next(address) for L in layers}
    r.chw = {L["name"]: next(address) for L in layers if L["op"] == "depthwise"}
    r._forget()
    return r


def small_table():
    """Depthwise + pointwise twice (a chain), a depthwise layer, two layers that read the input as well, a linear layer."""
    def bn(n):
        return dict(bias=np.zeros(n, np.int8), k=np.ones(n), lam=np.zeros(n), relu=1, bn=1, mult=0, shift=5)

    def dw(name, src):
        return dict(bn(64), op="depthwise", name=name, **{"in": src}, w=np.zeros((64, 3, 3), np.int8), pads=[1, 1, 1, 1], strides=[1, 1])

    def pw(name, src):
        return dict(bn(64), op="pointwise", name=name, **{"in": src}, w=np.zeros((64, 1, 1, 64), np.int8))

    return [dw("d1", "input"), pw("p1", "d1"), dw("d2", "p1"), pw("p2", "d2"), dw("d3", "p2"),
            dict(op="add", name="sum", **{"in": ("d3", "input")}, m1=1, m2=1, shift=1),
            dict(op="maxpool", name="pool", **{"in": "sum"}, kernel=[2, 2], strides=[2, 2], out_hw=[4, 4]),
            dict(bn(10), op="linear", name="fc", **{"in": "pool"}, w=np.zeros((10, 4 * 4 * 64), np.int8))]


def test_runner_falls_back_from_its_plan():
    """An input for which the library has no kernel (here: at an odd address) takes the layers that a walk takes for it, also
    once there is a plan; what has been queued is not queued again."""
    def odd_is_refused(lib):
        def on_call(n, name, pointers):
            if name in ("pulp_nn_hip_dw_pw_chain_hwc", "pulp_nn_hip_depthwise_hwc", "pulp_nn_hip_dw_pw_hwc") and pointers[0] % 4:
                lib.error = 2
                lib.seen.pop()
        lib.on_call = on_call

    whole, tail, behind = small_table(), small_table()[4:], small_table()[4:]
    tail[0]["in"] = behind[0]["in"] = "input"
    behind.insert(0, dict(op="add", name="twice", **{"in": ("input", "input")}, m1=1, m2=1, shift=1))
    behind[2]["in"] = ("d3", "twice")
    for table in (whole, tail, behind):   # the refused call is the first one, or not
        runs = []
        for xs in ((0x100, 0x200, 0x300, 0x301), (0x301,)):
            lib = FakeLibrary()
            odd_is_refused(lib)
            r = bare_runner(lib.bound(), table, (8, 8, 64))
            for x in xs:
                lib.seen.clear()
                out = r.run(x)
            assert out == r.act["fc"]
            runs.append((list(lib.seen), r.launches))
        assert runs[0] == runs[1] and len(set(runs[0][0])) == len(runs[0][0])
        assert any(name == "pulp_nn_depthwise_generic" for name, *_ in runs[0][0])


@pytest.mark.parametrize("how", ["subclass", "attribute", "class attribute", "chain", "wrapper"])
def test_overridden_methods_are_called_at_every_run(how, monkeypatch):
    """Tracing or logging put over a layer method, before the runner is made or once it has a plan; an object that only wraps
    a library."""
    lib, log = FakeLibrary(), []
    name = "dw_pw_chain_hwc" if how == "chain" else "pulp_nn_add"
    original = getattr(api.PulpNN, name)

    def traced(self, *args):
        log.append(args[0])
        return original(self, *args)

    if how == "wrapper":
        real = lib.bound()

        class Wrapper:
            def __getattr__(self, n):
                return getattr(real, n) if n != name else lambda *args: traced(real, *args)
        nn = Wrapper()
    else:
        nn = lib.bound(type("Traced", (api.PulpNN,), {name: traced}) if how == "subclass" else api.PulpNN)
    r = bare_runner(nn, small_table(), (8, 8, 64))
    if how not in ("subclass", "wrapper"):
        for x in (0x100, 0x200, 0x300):
            r.run(x)
        assert not log
    if how == "attribute":
        nn.pulp_nn_add = lambda *args: traced(nn, *args)
    elif how in ("class attribute", "chain"):
        monkeypatch.setattr(api.PulpNN, name, traced, raising=False)
    runs = []
    for x in (0x400, 0x500, 0x600):
        log.clear()
        lib.seen.clear()
        r.run(x)
        assert log == ([x] if how == "chain" else [r.act["d3"]])
        runs.append([c[1:] for c in lib.seen])
    assert [len(s) for s in runs] == [5] * 3
    if how == "attribute":               # and away again
        del nn.pulp_nn_add
        for x in (0x400, 0x500, 0x600):
            log.clear()
            r.run(x)
            assert not log


def test_runner_notices_every_change():
    """Whatever run() reads of the table, the parameters and the buffers: after a change, in place or not, and one run later
    the calls are those of a runner that has just been made."""
    def changes():
        yield lambda r: r.layers[0]["pads"].__setitem__(0, 2)
        yield lambda r: r.layers[2]["strides"].__setitem__(slice(None), [2, 2])
        yield lambda r: r.layers[6]["kernel"].__setitem__(1, 3)
        yield lambda r: r.layers[4].update(shift=7)
        yield lambda r: r.layers[4].update(mult=np.int32(3))
        yield lambda r: r.layers[5].update(m2=2)
        yield lambda r: r.layers[6].update(pads=(0, 1, 0, 0))     # a key that was absent
        yield lambda r: r.params[7].pop("bias")
        yield lambda r: r.params[1].update(bias=0x99)
        yield lambda r: r.params.__setitem__(3, dict(r.params[3], w=0x98))
        yield lambda r: r.act.update(sum=0x97)
        yield lambda r: r.shapes.update(fc=(1, 1, 9))
        yield lambda r: setattr(r, "fused", False)
        yield lambda r: r.unchained.add(0)

    def calls_of(r, lib):
        lib.seen.clear()
        r.run(0x100)
        return list(lib.seen)

    for i, change in enumerate(changes()):
        lib = FakeLibrary()
        original = network.Runner._walk
        r = bare_runner(lib.bound(), small_table(), (8, 8, 64))
        walks = []
        r._walk = lambda *a, **k: (walks.append(a[1]), original(r, *a, **k))[1]
        for _ in range(3):
            before = calls_of(r, lib)
        walks.clear()
        assert calls_of(r, lib) == before and not walks, "change %d: the plan runs" % i
        change(r)
        after = calls_of(r, lib)
        assert walks, "change %d was not noticed" % i
        assert calls_of(r, lib) == after and calls_of(r, lib) == after, "change %d" % i


def test_runner_keeps_no_plan_of_entries_that_change_without_a_trace():
    lib = FakeLibrary()
    r = bare_runner(lib.bound(), small_table(), (8, 8, 64))
    r.layers[6]["kernel"] = np.array([2, 2])
    for _ in range(4):
        r.run(0x100)
    assert r._plan is None
    r = bare_runner(lib.bound(), small_table(), (8, 8, 64))
    r.layers[4]["shift"] = np.int64(5)                            # immutable: a plan
    for _ in range(4):
        r.run(0x100)
    assert r._plan is not None


def test_the_first_run_lays_the_plan_out():
    """A new runner walks its table once: the calls go out during the first run, and the second run is the plan's."""
    lib, walks = FakeLibrary(), []
    r = bare_runner(lib.bound(), small_table(), (8, 8, 64))
    original = network.Runner._walk
    r._walk = lambda *a, **k: (walks.append(len(lib.seen)), original(r, *a, **k))[1]
    r.run(0x100)
    first = list(lib.seen)
    assert walks == [0] and len(first) == 5
    lib.seen.clear()
    assert r.run(0x200) == r.act["fc"] and len(walks) == 1 and r.launches == 5
    assert lib.seen == [tuple(0x200 if p == 0x100 else p for p in call) for call in first]
    # an input that is one of the runner's own buffers is told from the buffer
    r = bare_runner(lib.bound(), small_table(), (8, 8, 64))
    r.run(r.act["p2"])
    lib.seen.clear()
    r.run(0x300)
    assert lib.seen[0] == ("pulp_nn_hip_dw_pw_chain_hwc", 0x300, r.act["p2"], r.params[0]["w"], r.params[2]["w"])


def small_blocks():
    """Blocks on 16 x 16 planes: one that reads the input, one behind it."""
    def bn(n):
        return dict(bias=np.zeros(n, np.int8), k=np.ones(n), lam=np.zeros(n), relu=1, bn=1, mult=0, shift=5)

    def dw(name, src):
        return dict(bn(64), op="depthwise", name=name, **{"in": src}, w=np.zeros((64, 3, 3), np.int8), pads=[1, 1, 1, 1], strides=[1, 1])

    def pw(name, src, co):
        return dict(bn(co), op="pointwise", name=name, **{"in": src}, w=np.zeros((co, 1, 1, 64), np.int8))

    return [dw("d1", "input"), pw("p1", "d1", 64), dw("d2", "p1"), pw("p2", "d2", 32)]


def test_depthwise_results_of_small_blocks_can_be_read():
    """The rule that makes one launch of a small block: whoever reads the depthwise result, before or after the run, gets it as
    from the two launches."""
    def runner():
        lib = FakeLibrary()
        nn = lib.bound()
        nn._lib.pulp_nn_hip_get_batch = lambda: lib.batch
        r = bare_runner(nn, small_blocks(), (16, 16, 64), batch=4)
        r.act = network._Activations(r, r.act)
        return lib, r

    def calls(lib, r, x):
        lib.seen.clear()
        r.run(x)
        return [c[0].replace("pulp_nn_", "").replace("hip_", "") for c in lib.seen]

    two, one = ["depthwise_hwc", "pointwise_HoWo_parallel"], ["dw_pw_hwc"]
    readers = [lambda r: r.act["d2"], lambda r: r.act.get("d2"), lambda r: dict(r.act)["d2"], lambda r: {**r.act}["d2"],
               lambda r: list(r.act.values())[2], lambda r: dict(r.act.items())["d2"], lambda r: r.act.copy()["d2"],
               lambda r: r.act.setdefault("d2"), lambda r: copy.deepcopy(r.act)["d2"]]
    for read in readers:
        lib, r = runner()
        for x in (0x100, 0x200, 0x300):
            assert calls(lib, r, x) == two + one and r.launches == 3   # the input may be gone when d1 is read: two launches
        lib.seen.clear()
        lib.batch = 7                                     # (the caller's)
        buffer = read(r)
        assert buffer == dict.__getitem__(r.act, "d2") and lib.batch == 7
        assert [(c[0], c[1], c[3]) for c in lib.seen] == [("pulp_nn_hip_depthwise_hwc", dict.__getitem__(r.act, "p1"), buffer)]
        for x in (0x100, 0x200):
            assert calls(lib, r, x) == two + two and r.launches == 4
        lib.seen.clear()
        read(r)
        assert not lib.seen
    lib, r = runner()
    r.act["d2"]                                           # held from before the first run on
    assert calls(lib, r, 0x100) == two + two
    for put in (lambda r: r.act.__setitem__("d2", 0x990000), lambda r: r.act.update(d2=0x990000)):
        lib, r = runner()
        assert calls(lib, r, 0x100) == two + one
        put(r)                                            # a buffer of the caller's
        assert calls(lib, r, 0x100) == two + two and lib.seen[2][3] == 0x990000
    lib, r = runner()
    r.act = dict(r.act)                                   # and a dictionary that does not tell who reads it
    assert calls(lib, r, 0x100) == two + two


def test_blocks_of_two_branches_are_no_chain():
    """Two blocks of one shape, one after the other in the table, that read different tensors: each is called on its own input."""
    dw1, pw1, dw2, pw2 = small_table()[:4]
    pool = dict(op="maxpool", **{"in": "input"}, kernel=[2, 2], strides=[2, 2], out_hw=[8, 8])
    table = [dict(pool, name="a"), dict(pool, name="b"), dict(dw1, **{"in": "a"}), pw1, dict(dw2, **{"in": "b"}), pw2,
             dict(op="add", name="sum", **{"in": ("p1", "p2")}, m1=1, m2=1, shift=1)]
    lib = FakeLibrary()
    r = bare_runner(lib.bound(), table, (16, 16, 64))
    for x in (0x100, 0x200):
        lib.seen.clear()
        r.run(x)
        assert [c[0] for c in lib.seen][2:4] == ["pulp_nn_hip_dw_pw_hwc"] * 2 and len(lib.seen) == r.launches == 5
        assert [c[1] for c in lib.seen][2:4] == [r.act["a"], r.act["b"]] and [c[2] for c in lib.seen][2:4] == [r.act["p1"], r.act["p2"]]


def test_a_plan_does_not_keep_the_input():
    lib = FakeLibrary()
    r = bare_runner(lib.bound(), small_table(), (8, 8, 64))
    x = TensorLike(0x1000)
    before = sys.getrefcount(x)
    r.run(x)
    r.run(x)
    assert sys.getrefcount(x) == before


def in_a_new_process(code):
    res = subprocess.run([sys.executable, "-c", code], stdout=subprocess.PIPE, stderr=subprocess.PIPE, text=True, timeout=100,
                         cwd=os.path.dirname(os.path.dirname(os.path.abspath(__file__))))
    assert res.returncode == 0, res.stderr
    return res.stdout


def test_addresses_need_no_torch():
    """A caller that has raw addresses: torch is not needed where it cannot be imported."""
    code = ("import sys; sys.modules['torch'] = None\n"
            "from pulp_nn_amd import PulpNN, PulpNNError\n"
            "nn = PulpNN(32)\n"
            "try:\n    nn.pulp_nn_add(0, 0, 0, 1, 1, 1, 1, 1, 1)\n"
            "except PulpNNError as e:\n    print('code', e.code)\n")
    assert in_a_new_process(code) == "code 1\n"


def test_submodules_are_attributes_of_the_package():
    assert in_a_new_process("import pulp_nn_amd\nprint(pulp_nn_amd.build.__name__, pulp_nn_amd.api.__name__)") == "pulp_nn_amd.build pulp_nn_amd.api\n"


def test_binding_imported_before_the_build():
    """The extension is built after the binding was imported: PulpNN works from then on; before, the error names the file."""
    code = ("from pulp_nn_amd import api, build\n"
            "import os\n"
            "real = build.fast_path()\n"
            "api._fast, api.fast_path = None, lambda: '/nonexistent/_pulpnn_fast.so'\n"
            "source = open(api.__file__).read()\n"
            "build.fast_path = api.fast_path\n"
            "exec(compile(source, api.__file__, 'exec'), api.__dict__)\n"      # the binding as imported before the build
            "from pulp_nn_amd.api import PulpNN as early\n"
            "try:\n    early(32)\n"
            "except ImportError as e:\n    print('_pulpnn_fast.so is missing' in str(e))\n"
            "api.fast_path = build.fast_path = lambda: real\n"
            "a, b = early(32), early(64)\n"
            "print(a.bn_bits, b.bn_bits, type(a) is api.PulpNN, api.plain(a), early(32, check=False).check)\n")
    assert in_a_new_process(code) == "True\n32 64 True True False\n"
