"""A small layer-table format for chained int8 networks and a runner that executes it on the
GPU through the C API (what generated deployment code does by hand with the reference:
one pulp_nn_* call per layer on caller-owned buffers).

A network is a list of layer dicts.  Every layer has "op", "name" and "in" (the name of the
tensor it reads; the network input is called "input"; "add" takes a pair of names) and
produces the tensor called like the layer.  Activations are HWC uint8, batch outermost.

  op            parameters
  conv          w [Co,ky,kx,Ci] int8, bias [Co] int8 or None, pads (t,b,l,r), strides (sx,sy),
                requantisation (below)                      -> pulp_nn_conv_Ho_parallel
  pointwise     w [Co,1,1,Ci], bias, requantisation        -> pulp_nn_pointwise_HoWo_parallel
  depthwise     w [C,ky,kx], bias, pads, strides, requantisation.  The tensor it reads is HWC
                like all others; the runner changes the layout (pulp_nn_hip_hwc_to_chw +
                pulp_nn_depthwise_generic) or, for 3x3 / padding 1 layers the library has a
                fused kernel for, calls pulp_nn_hip_depthwise_hwc; if the next layer is a
                pointwise layer that is the only reader of the depthwise result, the two run
                as one launch (pulp_nn_hip_dw_pw_hwc) and the depthwise result is not
                materialised: Runner(..., fuse_blocks=True) for every such pair, False for none,
                "auto" (the default) where it is not slower: as Runner.tune() measured it on the
                batch at hand, else for blocks whose output plane is 8 x 8 pixels, small blocks, and
                blocks whose depthwise layer alone would need a layout change.  The depthwise
                results of the latter two can be had all the same: reading Runner.act computes them
                for the run before, and the runs after it make the two launches
  maxpool       kernel (kx,ky), strides, pads, out_hw      -> pulp_nn_maxpool
  avgpool       kernel, strides, pads, out_hw, lam, shift, add, requant -> pulp_nn_avgpool
  add           in = (a, b), m1, m2, shift                 -> pulp_nn_add
  linear        w [N,K] int8, bias, requantisation; reads its input flattened per image
                                                           -> pulp_nn_linear
  linear_out_32 w [N,K], bias32 [N] int32 or None; int32 output -> pulp_nn_linear_out_32

Requantisation keys: relu, bn (the two flags), k, lam ([Co] arrays for bn), mult (out_mult),
shift (out_shift).  shift = None on a bn layer means "to be calibrated": Runner.calibrate()
sets it to floor(log2(max |acc * k|)) - 7 over the batch it is given, computed on the GPU
(pulp_nn_hip_calib_conv / pulp_nn_hip_calib_depthwise), layer by layer along the chain.
"""
import collections.abc
import weakref

import numpy as np

from . import api
from .api import PulpNNError

_ARRAYS = frozenset(("w", "bias", "bias32", "k", "lam"))   # of a layer: uploaded once, not read by run()
CONV_LIKE = ("conv", "pointwise", "depthwise", "linear")


def out_size(n, k, s, p0, p1):
    return (n + p0 + p1 - k) // s + 1


def infer_shapes(layers, input_shape):
    """{tensor name: (H, W, C)} for the input and every layer output (linear outputs are (1, 1, N))."""
    shapes = {"input": tuple(input_shape)}
    for L in layers:
        op = L["op"]
        src = L["in"][0] if op == "add" else L["in"]
        H, W, Cc = shapes[src]
        if op in ("conv", "pointwise"):
            Co, ky, kx, Ci = L["w"].shape
            assert Ci == Cc, (L["name"], Ci, Cc)
            if op == "pointwise":
                shapes[L["name"]] = (H, W, Co)
            else:
                pt, pb, pl, pr = L["pads"]
                sx, sy = L["strides"]
                shapes[L["name"]] = L.get("out_hw", (out_size(H, ky, sy, pt, pb), out_size(W, kx, sx, pl, pr))) + (Co,)
        elif op == "depthwise":
            Cw, ky, kx = L["w"].shape
            assert Cw == Cc, (L["name"], Cw, Cc)
            pt, pb, pl, pr = L["pads"]
            sx, sy = L["strides"]
            shapes[L["name"]] = L.get("out_hw", (out_size(H, ky, sy, pt, pb), out_size(W, kx, sx, pl, pr))) + (Cc,)
        elif op in ("maxpool", "avgpool"):
            shapes[L["name"]] = tuple(L["out_hw"]) + (Cc,)
        elif op == "add":
            assert shapes[L["in"][1]] == (H, W, Cc), L["name"]
            shapes[L["name"]] = (H, W, Cc)
        elif op in ("linear", "linear_out_32"):
            N, K = L["w"].shape
            assert K == H * W * Cc, (L["name"], K, H * W * Cc)
            shapes[L["name"]] = (1, 1, N)
        else:
            raise ValueError("unknown op %r" % op)
    return shapes


class _Activations(dict):
    """Runner.act, {tensor name: buffer}: a tensor is handed out with the last run's values in it, also one that the run left
    out by the rule for small blocks; a buffer that the caller puts in its place is written by the next run."""

    def __init__(self, runner, buffers):
        super().__init__(buffers)
        self._runner = weakref.ref(runner)

    def __getitem__(self, name):
        runner = self._runner()
        if runner is not None and name in self:
            runner._hand_out(name)
        return super().__getitem__(name)

    def __setitem__(self, name, buffer):
        runner = self._runner()
        if runner is not None:
            runner._ask(name)
        super().__setitem__(name, buffer)

    def update(self, *args, **kwargs):
        for name, buffer in dict(*args, **kwargs).items():
            self[name] = buffer

    def __ior__(self, other):
        self.update(other)
        return self

    def get(self, name, default=None):
        return self[name] if name in self else default

    def values(self):
        return collections.abc.ValuesView(self)

    def items(self):
        return collections.abc.ItemsView(self)

    def pop(self, name, *default):
        if name in self:
            self[name]
        return super().pop(name, *default)

    def setdefault(self, name, default=None):
        return self[name] if name in self else super().setdefault(name, default)

    def __iter__(self):   # (its own, so that dict(act) and {**act} read the entries through __getitem__ too)
        return super().__iter__()

    def copy(self):
        return dict(self)

    def __reduce__(self):
        return dict, (dict(self),)


class Runner:
    """Uploads the parameters once, owns the activation buffers and queues the chain.

    The first run() walks the table in Python, learns which geometries have a fused kernel and lays the calls it made out as a
    plan (api's extension module); from then on a run() is one call that queues them, 2 us a launch instead of 9.  A plan belongs to the table and the buffers it was made from: a changed entry of a layer, of its parameters or of the
    buffers, a list changed in place, a changed choice makes run() walk again."""

    def __init__(self, nn, layers, input_shape, batch, fused=True, fuse_blocks="auto", chain_blocks=True):
        import torch
        self.nn, self.layers, self.batch, self.torch = nn, layers, batch, torch
        self.fused, self.unfused = fused, set()
        self.fuse_blocks, self.unfused_blocks, self.launches = fuse_blocks, set(), 0
        self.block_choice = {}   # layer index of a depthwise layer -> run it and its pointwise layer as one launch (tune())
        # runs of depthwise + pointwise blocks of one shape as one launch each (pulp_nn_hip_dw_pw_chain_hwc)
        self.chain_blocks, self.unchained = bool(chain_blocks and fused and fuse_blocks), set()
        self.shapes = infer_shapes(layers, input_shape)
        bn_np = np.int64 if nn.bn_bits == 64 else np.int32

        def dev(a, dtype=None):
            return None if a is None else torch.from_numpy(np.ascontiguousarray(a, dtype=dtype)).cuda()

        self.params = []
        for L in layers:
            P = {}
            if "w" in L:
                P["w"] = dev(L["w"], np.int8)
            if L["op"] == "linear_out_32":
                P["bias"] = dev(L.get("bias32"), np.int32)
            elif "bias" in L:
                P["bias"] = dev(L["bias"], np.int8)
            if L.get("k") is not None:
                P["k"], P["lam"] = dev(L["k"], bn_np), dev(L["lam"], bn_np)
            self.params.append(P)
        act = {}
        for L in layers:
            H, W, Cc = self.shapes[L["name"]]
            dt = torch.int32 if L["op"] == "linear_out_32" else torch.uint8
            act[L["name"]] = torch.empty((batch, H, W, Cc), dtype=dt, device="cuda")
        self.act = _Activations(self, act)
        self.chw = {}
        for L in layers:
            if L["op"] == "depthwise":
                H, W, Cc = self.shapes[L["in"]]
                self.chw[L["name"]] = torch.empty((batch, Cc, H, W), dtype=torch.uint8, device="cuda")
        self._calib = None
        self._forget()

    def _forget(self, plannable=True):
        self._plan = None        # (choices, objects, plan, result tensor, launches, [(layer, launches) before a call])
        self._plannable = plannable

    # -- buffers ----------------------------------------------------------------------------
    _asked = frozenset()     # depthwise layers (indices) whose results the caller has asked for
    _left_out = ()           # ... whose results the last run left out because their blocks are small

    def _buffer(self, name):
        return dict.__getitem__(self.act, name)

    def _ask(self, name):
        """Runs to come write tensor `name`; its layer's index, for a depthwise layer."""
        i = next((i for i, L in enumerate(self.layers) if L["name"] == name and L["op"] == "depthwise"), None)
        if i is not None:
            self._asked |= {i}
        return i

    def _hand_out(self, name):
        """The caller is given the buffer of tensor `name`: what the last run did not write into it is computed now."""
        i = self._ask(name)
        if i in self._left_out:
            src, batch = self.layers[i]["in"], self.nn.get_batch()
            self.nn.set_batch(self.batch)
            try:
                self._queue(i, {src: self._buffer(src)})
            finally:
                self.nn.set_batch(batch)

    # -- one layer ------------------------------------------------------------------------
    def _requant_args(self, L, P):
        relu, bn = L.get("relu", 0), L.get("bn", 0)
        if relu and bn and L.get("shift") is None:
            raise ValueError("layer %s has no out_shift: run calibrate() first" % L["name"])
        return P.get("k"), P.get("lam"), L.get("mult", 0), L.get("shift", 0) or 0, relu, bn

    def _queue(self, i, tensors, nn=None):
        L, P, nn = self.layers[i], self.params[i], nn or self.nn
        op, out = L["op"], self._buffer(L["name"])
        if op == "add":
            a, b = tensors[L["in"][0]], tensors[L["in"][1]]
            H, W, Cc = self.shapes[L["name"]]
            nn.pulp_nn_add(a, b, out, L["m1"], L["m2"], L["shift"], H, W, Cc)
            return out
        cur = tensors[L["in"]]
        H, W, Cc = self.shapes[L["in"]]
        Ho, Wo, Co = self.shapes[L["name"]]
        if op in ("conv", "pointwise"):
            k, lam, mult, shift, relu, bn = self._requant_args(L, P)
            if op == "conv":
                ky, kx = L["w"].shape[1:3]
                pt, pb, pl, pr = L["pads"]
                sx, sy = L["strides"]
                nn.pulp_nn_conv_Ho_parallel(cur, None, P.get("bias"), out, P["w"], k, lam, mult, shift, W, H, Cc, Wo, Ho,
                                            Co, kx, ky, pt, pb, pl, pr, sx, sy, relu, bn)
            else:
                nn.pulp_nn_pointwise_HoWo_parallel(cur, None, P.get("bias"), out, P["w"], k, lam, mult, shift, W, H, Cc,
                                                   Wo, Ho, Co, 1, 1, 0, 0, 0, 0, 1, 1, relu, bn)
        elif op == "depthwise":
            k, lam, mult, shift, relu, bn = self._requant_args(L, P)
            ky, kx = L["w"].shape[1:3]
            pt, pb, pl, pr = L["pads"]
            sx, sy = L["strides"]
            fusable = (ky, kx) == (3, 3) and tuple(L["pads"]) == (1, 1, 1, 1) and sx == sy
            if self.fused and fusable and i not in self.unfused:
                try:
                    nn.depthwise_hwc(cur, P.get("bias"), out, P["w"], k, lam, mult, shift, W, H, Cc, Wo, Ho, sx, relu, bn)
                    return out
                except PulpNNError as err:
                    if err.code != 2:
                        raise
                    self.unfused.add(i)    # no fused kernel for this geometry
            chw = self.chw[L["name"]]
            nn.hwc_to_chw(cur, chw, W, H, Cc)
            nn.pulp_nn_depthwise_generic(chw, None, P.get("bias"), out, P["w"], None, k, lam, mult, shift, W, H, Cc,
                                         Wo, Ho, Cc, kx, ky, pt, pb, pl, pr, sx, sy, relu, bn)
        elif op == "maxpool":
            kx, ky = L["kernel"]
            sx, sy = L["strides"]
            pt, pb, pl, pr = L.get("pads", (0, 0, 0, 0))
            nn.pulp_nn_maxpool(cur, out, W, H, Cc, Wo, Ho, kx, ky, pt, pb, pl, pr, sx, sy)
        elif op == "avgpool":
            kx, ky = L["kernel"]
            sx, sy = L["strides"]
            pt, pb, pl, pr = L.get("pads", (0, 0, 0, 0))
            nn.pulp_nn_avgpool(cur, out, L.get("lam", 0), L.get("shift", 0), L.get("add", 0), W, H, Cc, Wo, Ho, kx, ky,
                               pt, pb, pl, pr, sx, sy, L.get("requant", 0))
        elif op == "linear":
            k, lam, mult, shift, relu, bn = self._requant_args(L, P)
            nn.pulp_nn_linear(cur, P.get("bias"), out, P["w"], k, lam, mult, shift, H * W * Cc, Co, relu, bn)
        elif op == "linear_out_32":
            nn.pulp_nn_linear_out_32(cur, P.get("bias"), out, P["w"], H * W * Cc, Co)
        else:
            raise ValueError(op)
        return out

    def run(self, x):
        """x: device tensor batch,H,W,C uint8.  Queues every layer; returns the last layer's tensor."""
        if not api.plain(self.nn):   # a layer method is overridden, or nn only wraps a library: its methods are called
            self._forget()
            return self._walk(x, self.nn)
        choices, laid_out = self._choices(), self._plan
        if laid_out is not None:
            made_with, objects, plan, out, launches, calls_at = laid_out
            if made_with == choices and all(a is b for a, b in zip(objects, self._objects())):
                done = plan.run(x)
                if done is True:
                    self.launches = launches
                    return out
                if done is not False:   # no kernel for a call on this input (its alignment): the walk takes other layers from there
                    self._plan = None
                    return self._walk(x, self.nn, *calls_at[done])
            self._plan = None
        if not self._plannable or not self.layers or any(x is t for d in (self.act, self.chw) for t in dict.values(d)):
            return self._walk(x, self.nn)
        rec = api._fast.Recorder(self.nn, x)
        out = self._walk(x, rec)
        self._lay_out_plan(rec, out)
        return out

    def _choices(self):
        return (len(self.layers), len(self.params), self.batch, self.fused, self.fuse_blocks, self.chain_blocks, tuple(self.unfused),
                tuple(self.unfused_blocks), tuple(self.unchained), tuple(self.block_choice.items()), self._asked)

    def _objects(self):
        return (self.nn, self.layers, self.params, self.act, self.chw, self.shapes, *self.layers, *self.params)

    def _lay_out_plan(self, rec, out):
        """The calls of a walk and the entries they were made from."""
        try:
            plan = api._fast.Plan(self.nn, self.batch, rec.calls, rec.input,
                                  [(self.layers, _ARRAYS), (self.params, None), ([self.act, self.chw, self.shapes], None)])
        except Exception:   # (an entry that may change in place without a trace, for one: no plan, the calls are made)
            return self._forget(plannable=False)
        self._plan = (self._choices(), self._objects(), plan, out, self.launches, rec.calls_at)

    def _walk(self, x, nn, first=0, launches=0):
        """Queues the layers from `first` on, the ones before it being queued in `launches` launches."""
        nn.set_batch(self.batch)
        act, held = self.act, dict.__getitem__
        tensors = {"input": x, **{L["name"]: held(act, L["name"]) for L in self.layers[:first]}}
        out = x
        self.launches = launches
        left_out = self._left_out = [i for i in self._left_out if i < first]
        recorded, readers = nn is not self.nn, None
        i = first
        while i < len(self.layers):
            if recorded:
                nn.at = (i, self.launches)
            L = self.layers[i]
            block = L["op"] == "depthwise"
            if block and readers is None:
                readers = self._reader_counts()
            n = self._chain_length(i, readers) if block and self.chain_blocks else 0
            if n >= 2 and self._queue_chain(i, n, tensors, nn):
                last = self.layers[i + 2 * n - 1]["name"]
                out = tensors[last] = held(act, last)
                i += 2 * n
                continue
            if block:
                small = self._small(i)
                # (a run of one block is one that can be one launch)
                if (self._pays(i, small) if n else self._block_fusable(i, readers=readers, small=small)) and self._queue_block(i, tensors, nn):
                    name = self.layers[i + 1]["name"]
                    out = tensors[name] = held(act, name)
                    if small:
                        left_out.append(i)
                    i += 2
                    continue
            out = tensors[L["name"]] = self._queue(i, tensors, nn)
            self.launches += 2 if (L["op"] == "depthwise" and (not self.fused or i in self.unfused)) else 1
            i += 1
        return out

    # -- depthwise + pointwise as one launch ------------------------------------------------
    def _block_fusable(self, i, policy=True, readers=None, small=None):
        """Layer i is a 3x3 / padding 1 depthwise layer whose only reader is the pointwise layer i + 1.
        policy=False: only whether the block can be one launch, not whether it pays on its own.
        readers, small: _reader_counts() and _small(i), where the caller has them."""
        if not (self.fused and self.fuse_blocks) or i in self.unfused_blocks or i + 1 >= len(self.layers):
            return False
        L, N = self.layers[i], self.layers[i + 1]
        if L["op"] != "depthwise" or N["op"] != "pointwise" or N["in"] != L["name"]:
            return False
        if policy and not self._pays(i, small):
            return False
        sx, sy = L["strides"]
        if L["w"].shape[1:3] != (3, 3) or tuple(L["pads"]) != (1, 1, 1, 1) or sx != sy:
            return False
        return (readers or self._reader_counts())[L["name"]] == 1

    def _pays(self, i, small=None):
        """Whether a block that can be one launch is to be one.  small: _small(i), where the caller has it."""
        # "auto": where the single launch is not slower than the two.  Runner.tune() times both forms of every such block on
        # the batch at hand and records the faster one in block_choice.  Without that measurement: output planes of 8 x 8
        # pixels, a whole image per workgroup (two launches / one at batch 256: 16x16x128 -> 256 at stride 2 10.2 / 8.1 us,
        # 8x8x256 11.6 / 8.8), and small blocks
        if self.fuse_blocks != "auto":
            return True
        if i in self.block_choice:
            return self.block_choice[i]
        return (self._small(i) if small is None else small) or self.shapes[self.layers[i]["name"]][:2] == (8, 8)

    def _small(self, i):
        """Whether fuse_blocks="auto" makes one launch of depthwise layer i and the next because the block is small, or because
        the depthwise layer alone would be two launches itself.  Not where its result is asked for, or could not be computed
        again for a caller who asks after the run, from an input that may be gone by then."""
        # Small: launches and round trips to memory are most of the time.  Two launches / one: 16x16x128 at batch 16 9.1 / 5.7 us,
        # 4x4x512 at batch 64 9.5 / 9.3; 64x64x16 at batch 64 11.5 / 9.7, at batch 256 20.2 / 24.3; 32x32x64 at batch 64 10.3 / 7.8, at
        # batch 256 16.9 / 19.1; so at most 4 MB for planes of 32 x 32 pixels and more.  Smaller planes would gain up to some 4 MB
        # too (16x16x128 at batch 128 13.0 / 8.1), but tables of 1 MB and more keep the launches per layer that callers count on.
        # No kernel for HWC input: 64x64x16 at batch 255 39.0 / 24.5 us, three launches / one.
        L = self.layers[i]
        Ho, Wo, Cc = self.shapes[L["name"]]
        size = self.batch * Ho * Wo * Cc
        if not (size < 2 ** 20 or (size <= 2 ** 22 and Ho * Wo >= 1024) or
                (Cc % 64 != 0 and (self.shapes[L["in"]][1] <= 8 or (self.batch * Cc) % 64 != 0))):
            return False
        return not (Ho == Wo == 8 or self.fuse_blocks != "auto" or i in self.block_choice or i in self._asked or L["in"] == "input" or
                    not isinstance(self.act, _Activations))

    def _reader_counts(self):
        """{tensor name: how many layers read it}"""
        counts = {}
        for M in self.layers:
            for name in (set(M["in"]) if M["op"] == "add" else (M["in"],)):
                counts[name] = counts.get(name, 0) + 1
        return counts

    def _chain_length(self, i, readers=None):
        """How many depthwise + pointwise blocks of one shape start at layer i (stride 1, as many channels out as in,
        every intermediate tensor read by the next layer only): such a run is one launch, with the activations kept
        in LDS from block to block."""
        if i in self.unchained:
            return 0
        n, layers, shapes, shape = 0, self.layers, self.shapes, None
        readers = readers or self._reader_counts()
        while n < 8 and i + 2 * n + 1 < len(layers):
            L = layers[i + 2 * n]
            if L["op"] != "depthwise" or L["strides"][0] != 1 or (n > 0 and (L["in"] != layers[i + 2 * n - 1]["name"] or readers[L["in"]] != 1)):
                break
            shape = shape or shapes[L["in"]]
            if shapes[L["in"]] != shape or shapes[layers[i + 2 * n + 1]["name"]] != shape or \
                    not self._block_fusable(i + 2 * n, policy=False, readers=readers):
                break
            n += 1
        return n

    def _queue_chain(self, i, n, tensors, nn=None):
        nn = nn or self.nn
        H, W, Cc = self.shapes[self.layers[i]["in"]]
        blocks = []
        for j in range(n):
            L, P, N, Q = self.layers[i + 2 * j], self.params[i + 2 * j], self.layers[i + 2 * j + 1], self.params[i + 2 * j + 1]
            k1, l1, m1, s1, r1, b1 = self._requant_args(L, P)
            k2, l2, m2, s2, r2, b2 = self._requant_args(N, Q)
            blocks.append((P["w"], P.get("bias"), k1, l1, m1, s1, r1, b1, Q["w"], Q.get("bias"), k2, l2, m2, s2, r2, b2))
        try:
            nn.dw_pw_chain_hwc(tensors[self.layers[i]["in"]], self._buffer(self.layers[i + 2 * n - 1]["name"]), W, H, Cc, blocks)
        except PulpNNError as err:
            if err.code != 2:
                raise
            self.unchained.add(i)    # these blocks cannot share a launch
            return False
        self.launches += 1
        return True

    def _queue_block(self, i, tensors, nn=None):
        L, P, N, Q, nn = self.layers[i], self.params[i], self.layers[i + 1], self.params[i + 1], nn or self.nn
        H, W, Cc = self.shapes[L["in"]]
        Ho, Wo, Co = self.shapes[N["name"]]
        k1, l1, m1, s1, r1, b1 = self._requant_args(L, P)
        k2, l2, m2, s2, r2, b2 = self._requant_args(N, Q)
        try:
            nn.dw_pw_hwc(tensors[L["in"]], self._buffer(N["name"]), W, H, Cc, Wo, Ho, Co, L["strides"][0], P["w"], P.get("bias"),
                         k1, l1, m1, s1, r1, b1, Q["w"], Q.get("bias"), k2, l2, m2, s2, r2, b2)
        except PulpNNError as err:
            if err.code != 2:
                raise
            self.unfused_blocks.add(i)    # no fused kernel for this geometry
            return False
        self.launches += 1
        return True

    # -- calibration ------------------------------------------------------------------------
    def _calib_buffers(self):
        if self._calib is None:
            torch = self.torch
            most = max(self.batch * int(np.prod(self.shapes[L["name"]])) for L in self.layers)
            nbytes = self.nn.calib_workspace_bytes(most)
            self._calib = (torch.empty(nbytes // 8 + 1, dtype=torch.int64, device="cuda"), nbytes,
                           torch.zeros(2, dtype=torch.int64, device="cuda"))
        return self._calib

    def layer_absmax(self, i, tensors):
        """(max |acc * k|, derived out_shift) of conv-like layer i on the GPU."""
        L, P, nn = self.layers[i], self.params[i], self.nn
        ws, nbytes, res = self._calib_buffers()
        cur = tensors[L["in"]]
        H, W, Cc = self.shapes[L["in"]]
        Ho, Wo, Co = self.shapes[L["name"]]
        nn.set_batch(self.batch)
        if L["op"] == "depthwise":
            ky, kx = L["w"].shape[1:3]
            pt, _, pl, _ = L["pads"]
            sx, sy = L["strides"]
            nn.calib_depthwise(cur, P.get("bias"), P["w"], P["k"], W, H, Cc, Wo, Ho, kx, ky, pt, pl, sx, sy, 1, ws,
                               nbytes, res)
        elif L["op"] == "linear":
            nn.calib_conv(cur, P.get("bias"), P["w"], P["k"], 1, 1, H * W * Cc, 1, 1, Co, 1, 1, 0, 0, 1, 1, ws, nbytes, res)
        else:
            ky, kx = L["w"].shape[1:3]
            pt, _, pl, _ = L.get("pads", (0, 0, 0, 0))
            sx, sy = L.get("strides", (1, 1))
            nn.calib_conv(cur, P.get("bias"), P["w"], P["k"], W, H, Cc, Wo, Ho, Co, kx, ky, pt, pl, sx, sy, ws, nbytes, res)
        nn.sync()
        m, shift = (int(v) for v in res.cpu().numpy().view(np.uint64))
        if nn.bn_bits == 32 and m >= 2 ** 31:
            # the 32-bit tree forms acc * k in int32 (pulp_nn_utils.c:35-45): the layer's product wraps on this batch,
            # and no out_shift derived from the unwrapped maximum describes what the layer computes
            raise ValueError("layer %s: max |acc * k| = %d does not fit int32; the 32-bit batch-norm product wraps "
                             "(use smaller k or the 64-bit library)" % (L["name"], m))
        return m, shift

    def tune(self, x, reps=20):
        """Times every depthwise + pointwise block that can be one launch (and is not part of a chained run) both
        ways on this batch and keeps the faster form (fuse_blocks="auto" then follows these choices instead of the
        shape rule).  Needs every out_shift (run calibrate() first).  Returns {depthwise layer name: fused?}."""
        torch = self.torch
        self.nn.set_batch(self.batch)
        tensors = {"input": x}
        self.run(x)
        for L in self.layers:
            tensors[L["name"]] = self._buffer(L["name"])
        self.nn.sync()

        def timed(fn):
            fn()
            self.nn.sync()
            e0, e1 = torch.cuda.Event(enable_timing=True), torch.cuda.Event(enable_timing=True)
            e0.record()
            for _ in range(reps):
                fn()
            e1.record()
            self.nn.sync()
            return e0.elapsed_time(e1) / reps

        chosen = {}
        i = 0
        while i < len(self.layers):
            n = self._chain_length(i) if self.chain_blocks else 0
            if n >= 2:
                i += 2 * n
                continue
            if self._block_fusable(i, policy=False):
                ok = self._queue_block(i, tensors)   # False: the library has no fused kernel for this geometry
                if ok:
                    t_fused = timed(lambda: self._queue_block(i, tensors))
                    t_split = timed(lambda: (self._queue(i, tensors), self._queue(i + 1, tensors)))
                    self.block_choice[i] = t_fused <= t_split
                else:
                    self.block_choice[i] = False
                chosen[self.layers[i]["name"]] = self.block_choice[i]
                i += 2
                continue
            i += 1
        self.nn.sync()
        return chosen

    def calibrate(self, x, force=False):
        """Runs the chain on x and gives every batch-norm layer without an out_shift (all of them with
        force=True) the shift floor(log2(max |acc * k|)) - 7 measured on this batch.  Returns {name: shift}."""
        self.nn.set_batch(self.batch)
        tensors = {"input": x}
        chosen = {}
        for i, L in enumerate(self.layers):
            if L["op"] in CONV_LIKE and L.get("relu") and L.get("bn") and (force or L.get("shift") is None):
                _, L["shift"] = self.layer_absmax(i, tensors)
                chosen[L["name"]] = L["shift"]
            tensors[L["name"]] = self._queue(i, tensors)
        self.nn.sync()
        return chosen
