"""Python binding of libpulpnn_hip{32,64}.so (the C ABI declared in include/): the library is loaded with ctypes, the
layer functions are called through csrc/pybind_fast.cpp (argument conversion in C)."""
import ctypes as C
import importlib.machinery
import importlib.util
import os

from .build import fast_path, lib_path, tensor_path

_U16, _I8, _INT, _PTR = C.c_uint16, C.c_int8, C.c_int, C.c_void_p


def _load_fast():
    """The extension module, or None if it has not been built."""
    path = fast_path()
    if not os.path.exists(path):
        return None
    loader = importlib.machinery.ExtensionFileLoader("_pulpnn_fast", path)
    mod = importlib.util.module_from_spec(importlib.util.spec_from_loader("_pulpnn_fast", loader))
    loader.exec_module(mod)
    return mod


_MISSING = "%s is missing: build it with `python -m pulp_nn_amd.build` (there is no CPU fallback)"
_fast = _load_fast()


def _load_torch():
    """Before a library is loaded: torch, where there is one, brings the HIP runtime that both then share, and its tensors
    are told apart by _pulpnn_tensor.so.  Without torch the functions take addresses."""
    try:
        import torch  # noqa: F401
    except ImportError:
        return
    if not os.path.exists(tensor_path()):
        raise ImportError(_MISSING % tensor_path())
    lib = C.PyDLL(tensor_path())
    _fast.set_tensor_function(C.cast(lib.pulpnn_tensor_address, _PTR).value)


class HipBlock(C.Structure):
    """pulp_nn_hip_block of include/pulp_nn_hip.h: the parameters of one depthwise + pointwise block."""
    _fields_ = [("dw_wt", _PTR), ("dw_bias", _PTR), ("dw_k", _PTR), ("dw_lambda", _PTR),
                ("dw_out_mult", _U16), ("dw_out_shift", _U16), ("dw_flag_relu", _I8), ("dw_flag_batch_norm", _I8),
                ("pw_weight", _PTR), ("pw_bias", _PTR), ("pw_k", _PTR), ("pw_lambda", _PTR),
                ("pw_out_mult", _U16), ("pw_out_shift", _U16), ("pw_flag_relu", _I8), ("pw_flag_batch_norm", _I8)]

CONV_NAMES = ("pulp_nn_conv_Ho_parallel", "pulp_nn_conv_Co_parallel", "pulp_nn_conv_HoWo_parallel",
              "pulp_nn_pointwise_HoWo_parallel", "pulp_nn_pointwise_Ho_parallel", "pulp_nn_pointwise_Co_parallel")
DW_NAMES = ("pulp_nn_depthwise_generic", "pulp_nn_depthwise_generic_less_4_weights")

ERRORS = {0: "ok", 1: "argument", 2: "unsupported", 3: "runtime"}


class PulpNNError(RuntimeError):
    def __init__(self, code, msg):
        super().__init__("%s (%s)" % (msg, ERRORS.get(code, code)))
        self.code = code


def _ptr(x):
    """torch tensor / int / None -> device address."""
    if x is None:
        return None
    if isinstance(x, int):
        return x
    if not x.is_cuda:
        raise ValueError("PULP-NN HIP kernels take device tensors")
    if not x.is_contiguous():
        raise ValueError("tensor must be contiguous")
    return x.data_ptr()


FAST_NAMES = CONV_NAMES + DW_NAMES + (
    "pulp_nn_linear", "pulp_nn_linear_out_32", "pulp_nn_maxpool", "pulp_nn_avgpool", "pulp_nn_add", "pulp_nn_depthwise_3x3_s1",
    "pulp_nn_hip_hwc_to_chw", "pulp_nn_hip_depthwise_hwc", "pulp_nn_hip_dw_pw_hwc", "pulp_nn_hip_dw_pw_chain_hwc",
    "pulp_nn_hip_set_batch", "pulp_nn_hip_last_error")


class _Methods:
    """One loaded library (32- or 64-bit batch-norm parameters).

    With check=True (default) every layer call raises PulpNNError if the library
    rejected it; the C functions themselves return void like the reference's.

    The layer functions are methods of the base class, with the reference's names and argument lists (the four or so
    scalars of the added entry points in parentheses): pulp_nn_conv_{Ho,Co,HoWo}_parallel,
    pulp_nn_pointwise_{HoWo,Ho,Co}_parallel, pulp_nn_depthwise_generic, pulp_nn_depthwise_generic_less_4_weights,
    pulp_nn_depthwise_3x3_s1, pulp_nn_linear, pulp_nn_linear_out_32, pulp_nn_maxpool, pulp_nn_avgpool, pulp_nn_add;
    set_batch(n);
    hwc_to_chw(x, out, dim_x, dim_y, ch, pad_top=0, pad_bottom=0);
    depthwise_hwc(x, bias, out, wt, k, lam, out_mult, out_shift, dim_in_x, dim_in_y, ch, dim_out_x, dim_out_y, stride,
    flag_relu, flag_batch_norm): 3x3 depthwise, padding 1, HWC in and out (the layout change fused in); PulpNNError
    (unsupported) for geometries without a fused kernel;
    dw_pw_hwc(x, out, dim_in_x, dim_in_y, ch, dim_out_x, dim_out_y, ch_out, stride, dw_wt, dw_bias, dw_k, dw_lam, dw_mult,
    dw_shift, dw_relu, dw_bn, pw_w, pw_bias, pw_k, pw_lam, pw_mult, pw_shift, pw_relu, pw_bn): 3x3 depthwise (padding 1,
    HWC in) and the pointwise layer behind it in one launch; PulpNNError (unsupported) likewise."""

    def __init__(self, bn_bits=32, check=True):
        if bn_bits not in (32, 64):
            raise ValueError("bn_bits must be 32 or 64")
        path = lib_path(bn_bits)
        if not os.path.exists(path):
            raise ImportError(_MISSING % path)
        _load_torch()
        self.bn_bits = bn_bits
        self.check = bool(check)
        self.path = path
        L = self._lib = C.CDLL(path)
        self._bind(bn_bits, {n: C.cast(getattr(L, n), _PTR).value for n in FAST_NAMES})
        L.pulp_nn_matmul.argtypes = [_PTR, _PTR, _U16, _U16, _U16, _U16, _PTR, _PTR, _PTR, _PTR, _PTR, _INT, _INT]
        L.pulp_nn_matmul.restype = _PTR
        L.pulp_nn_hip_get_batch.restype = C.c_uint
        L.pulp_nn_hip_set_stream.argtypes = [_PTR]
        L.pulp_nn_hip_get_stream.restype = _PTR
        L.pulp_nn_hip_sync.restype = _INT
        L.pulp_nn_hip_clock_probe.argtypes = [_PTR]
        L.pulp_nn_hip_clock_probe.restype = None
        L.pulp_nn_hip_last_error.restype = _INT
        L.pulp_nn_hip_last_error_string.restype = C.c_char_p
        L.pulp_nn_hip_bn_bits.restype = _INT
        L.pulp_nn_hip_dw_pw_chain_hwc.argtypes = [_PTR] * 2 + [_U16] * 3 + [C.c_uint, C.POINTER(HipBlock)]
        L.pulp_nn_hip_dw_pw_chain_hwc.restype = None
        _U64 = C.c_uint64
        L.pulp_nn_hip_calib_workspace_bytes.argtypes, L.pulp_nn_hip_calib_workspace_bytes.restype = [_U64], _U64
        L.pulp_nn_hip_calib_conv.argtypes = [_PTR] * 4 + [_U16] * 12 + [_PTR, _U64, _PTR]
        L.pulp_nn_hip_calib_conv.restype = None
        L.pulp_nn_hip_calib_depthwise.argtypes = [_PTR] * 4 + [_U16] * 11 + [_INT, _PTR, _U64, _PTR]
        L.pulp_nn_hip_calib_depthwise.restype = None
        L.pulp_nn_hip_calib_conv_static.argtypes = [_PTR] * 4 + [_U16] * 12 + [_PTR]
        L.pulp_nn_hip_calib_conv_static.restype = None
        assert L.pulp_nn_hip_bn_bits() == bn_bits

    # -- added entry points ------------------------------------------------
    def get_batch(self):
        return int(self._lib.pulp_nn_hip_get_batch())

    def set_stream(self, stream):
        """stream: a torch.cuda.Stream, a raw hipStream_t address, or None (default stream)."""
        h = getattr(stream, "cuda_stream", stream)
        self._lib.pulp_nn_hip_set_stream(h if h else None)

    def use_torch_stream(self):
        import torch
        self.set_stream(torch.cuda.current_stream())

    def sync(self):
        rc = self._lib.pulp_nn_hip_sync()
        if rc:
            self._raise()

    def clock_probe(self, out):
        """Queues the 20 us clock probe; out: device tensor of two int64 (wall-clock ticks at 100 MHz, shader cycles)."""
        self._call("pulp_nn_hip_clock_probe", _ptr(out))

    def last_error(self):
        return int(self._lib.pulp_nn_hip_last_error())

    def last_error_string(self):
        return self._lib.pulp_nn_hip_last_error_string().decode()

    def clear_error(self):
        self._lib.pulp_nn_hip_clear_error()

    def _raise(self):
        code, msg = self.last_error(), self.last_error_string()
        self.clear_error()
        raise PulpNNError(code, msg)

    def _call(self, name, *args):
        res = getattr(self._lib, name)(*args)
        if self.check and self._lib.pulp_nn_hip_last_error():
            self._raise()
        return res

    def dw_pw_chain_hwc(self, x, out, dim_x, dim_y, ch, blocks):
        """Several depthwise + pointwise blocks of one shape (stride 1, ch channels throughout) in one launch.
        blocks: a list of tuples (dw_wt, dw_bias, dw_k, dw_lam, dw_mult, dw_shift, dw_relu, dw_bn, pw_w, pw_bias,
        pw_k, pw_lam, pw_mult, pw_shift, pw_relu, pw_bn), the arguments dw_pw_hwc takes per block.  Raises PulpNNError
        (unsupported) where the blocks cannot be chained."""
        arr = (HipBlock * len(blocks))()
        for dst, b in zip(arr, blocks):
            (dst.dw_wt, dst.dw_bias, dst.dw_k, dst.dw_lambda) = [_ptr(v) for v in b[0:4]]
            (dst.dw_out_mult, dst.dw_out_shift, dst.dw_flag_relu, dst.dw_flag_batch_norm) = b[4:8]
            (dst.pw_weight, dst.pw_bias, dst.pw_k, dst.pw_lambda) = [_ptr(v) for v in b[8:12]]
            (dst.pw_out_mult, dst.pw_out_shift, dst.pw_flag_relu, dst.pw_flag_batch_norm) = b[12:16]
        self._call("pulp_nn_hip_dw_pw_chain_hwc", _ptr(x), _ptr(out), dim_x, dim_y, ch, len(blocks), arr)

    # -- calibration ---------------------------------------------------------
    def calib_workspace_bytes(self, n_outputs):
        return int(self._lib.pulp_nn_hip_calib_workspace_bytes(int(n_outputs)))

    def calib_conv(self, x, bias, w, k, dim_in_x, dim_in_y, ch_in, dim_out_x, dim_out_y, ch_out, kx, ky, pad_top,
                   pad_left, stride_x, stride_y, workspace, workspace_bytes, result):
        """result (device, 2 x uint64) <- max |acc * k|, and the out_shift floor(log2(max)) - 7 derived from it."""
        self._call("pulp_nn_hip_calib_conv", _ptr(x), _ptr(bias), _ptr(w), _ptr(k), dim_in_x, dim_in_y, ch_in,
                   dim_out_x, dim_out_y, ch_out, kx, ky, pad_top, pad_left, stride_x, stride_y, _ptr(workspace),
                   int(workspace_bytes), _ptr(result))

    def calib_depthwise(self, x, bias, wt, k, dim_in_x, dim_in_y, ch, dim_out_x, dim_out_y, kx, ky, pad_top, pad_left,
                        stride_x, stride_y, input_is_hwc, workspace, workspace_bytes, result):
        self._call("pulp_nn_hip_calib_depthwise", _ptr(x), _ptr(bias), _ptr(wt), _ptr(k), dim_in_x, dim_in_y, ch,
                   dim_out_x, dim_out_y, kx, ky, pad_top, pad_left, stride_x, stride_y, int(input_is_hwc),
                   _ptr(workspace), int(workspace_bytes), _ptr(result))

    def calib_conv_static(self, x, bias, w, k, dim_in_x, dim_in_y, ch_in, dim_out_x, dim_out_y, ch_out, kx, ky,
                          pad_top, pad_left, stride_x, stride_y, result):
        """calib_conv without a workspace argument: the library's fixed scratch array holds the partial maxima."""
        self._call("pulp_nn_hip_calib_conv_static", _ptr(x), _ptr(bias), _ptr(w), _ptr(k), dim_in_x, dim_in_y, ch_in,
                   dim_out_x, dim_out_y, ch_out, kx, ky, pad_top, pad_left, stride_x, stride_y, _ptr(result))

    # -- the reference's inner two-pixel matmul (the layer functions are the base class's) ----
    def pulp_nn_matmul(self, pWeight, pIn, ch_out, num_col_im2col, out_shift, out_mult, k, lam, bias, pOut, pOut2,
                       flag_relu, flag_batch_norm):
        return self._call("pulp_nn_matmul", _ptr(pWeight), _ptr(pIn), int(ch_out), int(num_col_im2col),
                          int(out_shift) & 0xFFFF, int(out_mult) & 0xFFFF, _ptr(k), _ptr(lam), _ptr(bias), _ptr(pOut),
                          _ptr(pOut2), int(flag_relu), int(flag_batch_norm))


def _define():
    """PulpNN: the methods above on the extension module's base class."""
    global PulpNN, _METHODS
    PulpNN = type("PulpNN", (_Methods, _fast.Base), {"__doc__": _Methods.__doc__, "__module__": __name__})
    # {name: attribute} of what a run over a table calls
    names = ("set_batch", "hwc_to_chw", "depthwise_hwc", "dw_pw_hwc", "dw_pw_chain_hwc", "_call", "__getattribute__",
             *(n for n in FAST_NAMES if "_hip_" not in n))
    _METHODS = {n: next(vars(c)[n] for c in PulpNN.__mro__ if n in vars(c)) for n in names}


def plain(nn):
    """Whether nn's layer methods are PulpNN's own, so that a plan, which calls the library directly, does what they would do."""
    return _fast is not None and _fast.plain(nn, _METHODS)


if _fast is not None:
    _define()
else:
    class PulpNN:  # noqa: F811
        """Stands in until the extension module has been built, which may happen in this process."""

        def __new__(cls, *args, **kwargs):
            global _fast
            _fast = _fast or _load_fast()
            if _fast is None:
                raise ImportError(_MISSING % fast_path())
            if PulpNN is cls:
                _define()
            return PulpNN(*args, **kwargs)
