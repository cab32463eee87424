// The Python front end's call path: argument conversion and the call itself in C, for one loaded library.
//
// A layer of a few MB takes the GPU 4 to 7 us.  Through ctypes a call costs 3.5 us of argument conversion (25 Python
// objects, six of them tensors asked for their address) before hipLaunchKernel is reached; here it is a few tenths of a
// microsecond.  `Base` is the base class of api.PulpNN: its methods take the reference's argument lists.  `Recorder` makes
// such calls and keeps them.  `Plan` is a list of such calls with their arguments converted once, for a chain of layers on buffers that its owner keeps: a run
// is one Python call, and only the chain's input is converted per run.
//
// The entry points are looked up by ctypes (api.py loads the library) and handed over as addresses, so this module does
// not link against either library.  Nor against torch: what a tensor's address is says a function of _pulpnn_tensor.so
// (pybind_tensor.cpp), handed over where torch can be imported.
#define PY_SSIZE_T_CLEAN
#include <Python.h>
#include <structmember.h>

#include <stdint.h>
#include <string.h>

#include <exception>
#include <new>
#include <string>
#include <vector>

#include "../../include/pulp_nn_hip.h"

namespace {

typedef unsigned short u16;
typedef signed char i8;

enum Kind { CONV, DW, LINEAR, LINEAR32, MAXPOOL, AVGPOOL, ADD, DW3, HWC2CHW, DWHWC, DWPW, CHAIN, NKIND };

// argument types in order: p = tensor / address / None, i = what int() takes, n = an integer; names for keyword calls
// (null: positional only); the last `optional` arguments default to zero / null
struct KindInfo {
  const char *spec;
  const char *names;
  int optional;
};
const KindInfo kinds[NKIND] = {
    {"pppppppiiiiiiiiiiiiiiiiii", nullptr, 0},
    {"ppppppppiiiiiiiiiiiiiiiiii", nullptr, 0},
    {"ppppppiiiiii", "pIn bias pOut pWeights k lam out_mult out_shift dim_vec num_o_neurons flag_relu flag_batch_norm", 0},
    {"ppppii", "pIn bias pOut pWeights dim_vec num_o_neurons", 0},
    {"ppiiiiiiiiiiiii", nullptr, 0},
    {"ppiiiiiiiiiiiiiiiii", nullptr, 0},
    {"pppiiiiii", "in1 in2 out out_mult1 out_mult2 out_shift dim_h dim_w ch", 0},
    {"ppiiiiipiippiip", "In_Img Out_Img R C_ CH p_l p_r Kernel out_shift out_mult kappa lam flag_relu flag_batch_norm memory_chan", 1},
    {"ppnnnnn", "x out dim_x dim_y ch pad_top pad_bottom", 2},
    {"ppppppnnnnnnnnnn", "x bias out wt k lam out_mult out_shift dim_in_x dim_in_y ch dim_out_x dim_out_y stride flag_relu flag_batch_norm", 0},
    {"ppnnnnnnnppppnnnnppppnnnn",
     "x out dim_in_x dim_in_y ch dim_out_x dim_out_y ch_out stride dw_wt dw_bias dw_k dw_lam dw_mult dw_shift dw_relu dw_bn pw_w pw_bias pw_k "
     "pw_lam pw_mult pw_shift pw_relu pw_bn",
     0},
    {nullptr, nullptr, 0},
};

// entry points by index: the two families with several names first
enum Fn {
  F_CONV_HO, F_CONV_CO, F_CONV_HOWO, F_PW_HOWO, F_PW_HO, F_PW_CO, F_DW_GENERIC, F_DW_LESS4, F_LINEAR, F_LINEAR32, F_MAXPOOL,
  F_AVGPOOL, F_ADD, F_DW3, F_HWC2CHW, F_DWHWC, F_DWPW, F_CHAIN, F_SET_BATCH, F_LAST_ERROR, NFN
};
const char *fn_names[NFN] = {
    "pulp_nn_conv_Ho_parallel", "pulp_nn_conv_Co_parallel", "pulp_nn_conv_HoWo_parallel", "pulp_nn_pointwise_HoWo_parallel",
    "pulp_nn_pointwise_Ho_parallel", "pulp_nn_pointwise_Co_parallel", "pulp_nn_depthwise_generic",
    "pulp_nn_depthwise_generic_less_4_weights", "pulp_nn_linear", "pulp_nn_linear_out_32", "pulp_nn_maxpool", "pulp_nn_avgpool",
    "pulp_nn_add", "pulp_nn_depthwise_3x3_s1", "pulp_nn_hip_hwc_to_chw", "pulp_nn_hip_depthwise_hwc", "pulp_nn_hip_dw_pw_hwc",
    "pulp_nn_hip_dw_pw_chain_hwc", "pulp_nn_hip_set_batch", "pulp_nn_hip_last_error"};
const Kind fn_kind[F_SET_BATCH] = {CONV, CONV, CONV, CONV, CONV, CONV, DW, DW, LINEAR, LINEAR32, MAXPOOL, AVGPOOL, ADD, DW3, HWC2CHW, DWHWC, DWPW, CHAIN};

struct Base {
  PyObject_HEAD
  void *fn[NFN];
  int bits;
  char check;
};

struct Args {
  void *p[10];
  int64_t s[20];
};

// an object with a tensor's methods -> device address
bool other_ptr(PyObject *o, void **out)
{
  static const char *const asked[2] = {"is_cuda", "is_contiguous"};
  static const char *const refusal[2] = {"PULP-NN HIP kernels take device tensors", "tensor must be contiguous"};
  for (int i = 0; i < 2; i++) {
    PyObject *v = i ? PyObject_CallMethod(o, asked[i], nullptr) : PyObject_GetAttrString(o, asked[i]);
    if (!v) return false;
    const int yes = PyObject_IsTrue(v);
    Py_DECREF(v);
    if (yes < 0) return false;
    if (!yes) {
      PyErr_SetString(PyExc_ValueError, refusal[i]);
      return false;
    }
  }
  PyObject *v = PyObject_CallMethod(o, "data_ptr", nullptr);
  if (!v) return false;
  *out = PyLong_AsVoidPtr(v);
  Py_DECREF(v);
  return *out || !PyErr_Occurred();
}

// 1 and the tensor's address, 0 if the object is no tensor, -1 with an exception set; null without torch
int (*tensor_address)(PyObject *, void **) = nullptr;

// tensor / address / None -> device address
bool to_ptr(PyObject *o, void **out)
{
  if (o == Py_None) {
    *out = nullptr;
    return true;
  }
  if (!PyLong_Check(o)) {
    const int is = tensor_address ? tensor_address(o, out) : 0;
    return is ? is > 0 : other_ptr(o, out);
  }
  *out = PyLong_AsVoidPtr(o);
  return *out || !PyErr_Occurred();
}

bool to_int(PyObject *o, int64_t *out)
{
  if (PyLong_CheckExact(o)) {
    *out = (int64_t)PyLong_AsUnsignedLongLongMask(o);
    return true;
  }
  PyObject *n = PyNumber_Long(o);  // what int() accepts
  if (!n) return false;
  *out = (int64_t)PyLong_AsUnsignedLongLongMask(n);
  Py_DECREF(n);
  return true;
}

bool to_integer(PyObject *o, int64_t *out)
{
  if (PyLong_CheckExact(o)) return to_int(o, out);
  PyObject *n = PyNumber_Index(o);
  if (!n) return false;
  *out = (int64_t)PyLong_AsUnsignedLongLongMask(n);
  Py_DECREF(n);
  return true;
}

bool parse(Kind kind, PyObject *const *args, Py_ssize_t n, Args *a)
{
  const char *spec = kinds[kind].spec;
  const Py_ssize_t want = (Py_ssize_t)strlen(spec);
  if (n > want || n < want - kinds[kind].optional) {
    // (the functions without names have as many scalars as the reference's, which is asserted)
    const Py_ssize_t pointers = (Py_ssize_t)strspn(spec, "p");
    PyErr_Format(kinds[kind].names || n < pointers ? PyExc_TypeError : PyExc_AssertionError, "expected %zd arguments, got %zd", want, n);
    return false;
  }
  int np = 0, ns = 0;
  for (Py_ssize_t i = 0; i < want; i++) {
    if (spec[i] == 'p') {
      a->p[np] = nullptr;
      if (i < n && !to_ptr(args[i], &a->p[np])) return false;
      np++;
    } else {
      a->s[ns] = 0;
      if (i < n && !(spec[i] == 'i' ? to_int(args[i], &a->s[ns]) : to_integer(args[i], &a->s[ns]))) return false;
      ns++;
    }
  }
  return true;
}

#define U(i) (u16) a.s[i]
#define I(i) (int)a.s[i]
#define B8(i) (i8) a.s[i]
typedef void *P;

void invoke(const Base *b, int f, const Args &a, const pulp_nn_hip_block *blocks, unsigned n_blocks)
{
  void *fn = b->fn[f];
  void *const *p = a.p;
  switch (fn_kind[f]) {
    case CONV:
      ((void (*)(P, P, P, P, P, P, P, u16, u16, u16, u16, u16, u16, u16, u16, u16, u16, u16, u16, u16, u16, u16, u16, int, int))fn)(
          p[0], p[1], p[2], p[3], p[4], p[5], p[6], U(0), U(1), U(2), U(3), U(4), U(5), U(6), U(7), U(8), U(9), U(10), U(11), U(12),
          U(13), U(14), U(15), I(16), I(17));
      break;
    case DW:
      ((void (*)(P, P, P, P, P, P, P, P, u16, u16, u16, u16, u16, u16, u16, u16, u16, u16, u16, u16, u16, u16, u16, u16, i8, i8))fn)(
          p[0], p[1], p[2], p[3], p[4], p[5], p[6], p[7], U(0), U(1), U(2), U(3), U(4), U(5), U(6), U(7), U(8), U(9), U(10), U(11),
          U(12), U(13), U(14), U(15), B8(16), B8(17));
      break;
    case LINEAR:
      ((void (*)(P, P, P, P, P, P, u16, i8, u16, u16, int, int))fn)(p[0], p[1], p[2], p[3], p[4], p[5], U(0), B8(1), U(2), U(3), I(4), I(5));
      break;
    case LINEAR32: ((void (*)(P, P, P, P, u16, u16))fn)(p[0], p[1], p[2], p[3], U(0), U(1)); break;
    case MAXPOOL:
      ((void (*)(P, P, u16, u16, u16, u16, u16, u16, u16, u16, u16, u16, u16, u16, u16))fn)(
          p[0], p[1], U(0), U(1), U(2), U(3), U(4), U(5), U(6), U(7), U(8), U(9), U(10), U(11), U(12));
      break;
    case AVGPOOL:
      if (b->bits == 64)
        ((void (*)(P, P, int64_t, u16, int64_t, u16, u16, u16, u16, u16, u16, u16, u16, u16, u16, u16, u16, u16, int))fn)(
            p[0], p[1], a.s[0], U(1), a.s[2], U(3), U(4), U(5), U(6), U(7), U(8), U(9), U(10), U(11), U(12), U(13), U(14), U(15), I(16));
      else
        ((void (*)(P, P, int32_t, u16, int32_t, u16, u16, u16, u16, u16, u16, u16, u16, u16, u16, u16, u16, u16, int))fn)(
            p[0], p[1], I(0), U(1), I(2), U(3), U(4), U(5), U(6), U(7), U(8), U(9), U(10), U(11), U(12), U(13), U(14), U(15), I(16));
      break;
    case ADD: ((void (*)(P, P, P, u16, u16, u16, u16, u16, u16))fn)(p[0], p[1], p[2], U(0), U(1), U(2), U(3), U(4), U(5)); break;
    case DW3:
      ((void (*)(P, P, int, int, int, int, int, P, i8, u16, P, P, int, int, P))fn)(p[0], p[1], I(0), I(1), I(2), I(3), I(4), p[2], B8(5), U(6),
                                                                              p[3], p[4], I(7), I(8), p[5]);
      break;
    case HWC2CHW:
      ((void (*)(P, P, unsigned, unsigned, unsigned, unsigned, unsigned))fn)(p[0], p[1], (unsigned)a.s[0], (unsigned)a.s[1], (unsigned)a.s[2],
                                                                          (unsigned)a.s[3], (unsigned)a.s[4]);
      break;
    case DWHWC:
      ((void (*)(P, P, P, P, P, P, u16, u16, u16, u16, u16, u16, u16, u16, i8, i8))fn)(p[0], p[1], p[2], p[3], p[4], p[5], U(0), U(1), U(2), U(3),
                                                                                  U(4), U(5), U(6), U(7), B8(8), B8(9));
      break;
    case DWPW:
      ((void (*)(P, P, u16, u16, u16, u16, u16, u16, u16, P, P, P, P, u16, u16, i8, i8, P, P, P, P, u16, u16, i8, i8))fn)(
          p[0], p[1], U(0), U(1), U(2), U(3), U(4), U(5), U(6), p[2], p[3], p[4], p[5], U(7), U(8), B8(9), B8(10), p[6], p[7], p[8], p[9], U(11),
          U(12), B8(13), B8(14));
      break;
    case CHAIN:
      ((void (*)(P, P, u16, u16, u16, unsigned, const pulp_nn_hip_block *))fn)(p[0], p[1], U(0), U(1), U(2), n_blocks, blocks);
      break;
    default: break;
  }
}

int last_error(const Base *b) { return ((int (*)(void))b->fn[F_LAST_ERROR])(); }

// whether __init__ has looked the entry points up (all of them or none)
bool bound(const Base *b)
{
  if (!b->fn[F_LAST_ERROR]) PyErr_SetString(PyExc_RuntimeError, "library not bound");
  return b->fn[F_LAST_ERROR] != nullptr;
}

// keyword arguments -> their places (null: left out)
bool place_keywords(Kind kind, PyObject *const *args, Py_ssize_t n, PyObject *kw, std::vector<PyObject *> *out)
{
  const char *names = kinds[kind].names;
  if (!names) {
    PyErr_SetString(PyExc_TypeError, "this function takes no keyword arguments");
    return false;
  }
  std::vector<std::string> list;
  for (const char *s = names; *s;) {
    const char *e = strchr(s, ' ');
    list.emplace_back(s, e ? (size_t)(e - s) : strlen(s));
    s = e ? e + 1 : s + strlen(s);
  }
  out->assign(list.size(), nullptr);
  for (Py_ssize_t i = 0; i < n && i < (Py_ssize_t)list.size(); i++) (*out)[i] = args[i];
  for (Py_ssize_t j = 0; j < PyTuple_GET_SIZE(kw); j++) {
    const char *key = PyUnicode_AsUTF8(PyTuple_GET_ITEM(kw, j));
    size_t i = 0;
    while (i < list.size() && list[i] != key) i++;
    if (i == list.size() || (*out)[i]) {
      PyErr_Format(PyExc_TypeError, "unexpected or repeated argument '%s'", key);
      return false;
    }
    (*out)[i] = args[n + j];
  }
  while (!out->empty() && !out->back() && (int)(list.size() - out->size()) < kinds[kind].optional) out->pop_back();
  for (size_t i = 0; i < out->size(); i++)
    if (!(*out)[i]) {
      if (i + kinds[kind].optional < list.size()) {
        PyErr_Format(PyExc_TypeError, "missing argument '%s'", list[i].c_str());
        return false;
      }
    }
  return true;
}

template <int F>
PyObject *method(PyObject *self, PyObject *const *args, Py_ssize_t n, PyObject *kw)
{
  Base *b = (Base *)self;
  Args a;
  std::vector<PyObject *> placed;
  if (kw && PyTuple_GET_SIZE(kw)) {
    if (!place_keywords(fn_kind[F], args, n, kw, &placed)) return nullptr;
    // (an omitted optional argument in the middle: zero)
    static PyObject *zero = PyLong_FromLong(0);
    for (size_t i = 0; i < placed.size(); i++)
      if (!placed[i]) placed[i] = kinds[fn_kind[F]].spec[i] == 'p' ? Py_None : zero;
    args = placed.data();
    n = (Py_ssize_t)placed.size();
  }
  if (!bound(b)) return nullptr;
  if (!parse(fn_kind[F], args, n, &a)) return nullptr;
  int err;
  Py_BEGIN_ALLOW_THREADS
  invoke(b, F, a, nullptr, 0);
  err = b->check ? last_error(b) : 0;
  Py_END_ALLOW_THREADS
  if (err) return PyObject_CallMethod(self, "_raise", nullptr);
  Py_RETURN_NONE;
}

PyObject *set_batch(PyObject *self, PyObject *arg)
{
  int64_t v;
  if (!bound((Base *)self)) return nullptr;
  if (!to_int(arg, &v)) return nullptr;
  ((void (*)(unsigned))((Base *)self)->fn[F_SET_BATCH])((unsigned)v);
  Py_RETURN_NONE;
}

// _bind(bits, {name: address})
PyObject *bind(PyObject *self, PyObject *args)
{
  Base *b = (Base *)self;
  PyObject *d;
  if (!PyArg_ParseTuple(args, "iO!", &b->bits, &PyDict_Type, &d)) return nullptr;
  void *fn[NFN];
  for (int f = 0; f < NFN; f++) {
    PyObject *v = PyDict_GetItemString(d, fn_names[f]);
    if (!v) return PyErr_Format(PyExc_KeyError, "%s", fn_names[f]);
    fn[f] = PyLong_AsVoidPtr(v);
    if (PyErr_Occurred()) return nullptr;
  }
  memcpy(b->fn, fn, sizeof fn);
  Py_RETURN_NONE;
}

#define M(F, NAME) {NAME, (PyCFunction)(void (*)(void))method<F>, METH_FASTCALL | METH_KEYWORDS, nullptr}
PyMethodDef base_methods[] = {
    M(F_CONV_HO, "pulp_nn_conv_Ho_parallel"),
    M(F_CONV_CO, "pulp_nn_conv_Co_parallel"),
    M(F_CONV_HOWO, "pulp_nn_conv_HoWo_parallel"),
    M(F_PW_HOWO, "pulp_nn_pointwise_HoWo_parallel"),
    M(F_PW_HO, "pulp_nn_pointwise_Ho_parallel"),
    M(F_PW_CO, "pulp_nn_pointwise_Co_parallel"),
    M(F_DW_GENERIC, "pulp_nn_depthwise_generic"),
    M(F_DW_LESS4, "pulp_nn_depthwise_generic_less_4_weights"),
    M(F_LINEAR, "pulp_nn_linear"),
    M(F_LINEAR32, "pulp_nn_linear_out_32"),
    M(F_MAXPOOL, "pulp_nn_maxpool"),
    M(F_AVGPOOL, "pulp_nn_avgpool"),
    M(F_ADD, "pulp_nn_add"),
    M(F_DW3, "pulp_nn_depthwise_3x3_s1"),
    M(F_HWC2CHW, "hwc_to_chw"),
    M(F_DWHWC, "depthwise_hwc"),
    M(F_DWPW, "dw_pw_hwc"),
    {"set_batch", set_batch, METH_O, nullptr},
    {"_bind", bind, METH_VARARGS, nullptr},
    {nullptr, nullptr, 0, nullptr}};
PyObject *get_check(PyObject *self, void *) { return PyBool_FromLong(((Base *)self)->check); }
int set_check(PyObject *self, PyObject *value, void *)
{
  const int yes = value ? PyObject_IsTrue(value) : 0;
  if (yes < 0) return -1;
  ((Base *)self)->check = (char)yes;
  return 0;
}
PyGetSetDef base_getset[] = {{"check", get_check, set_check, "raise PulpNNError when the library rejects a call", nullptr},
                             {nullptr, nullptr, nullptr, nullptr, nullptr}};
PyTypeObject BaseType = {PyVarObject_HEAD_INIT(nullptr, 0)};

// ---- Recorder -----------------------------------------------------------------------------------------------------------

// Recorder(nn, x): stands in for nn during a walk over a table.  Makes the calls and keeps those that the library took, as Plan
// takes them: `calls`, with `input` in the place of x (an address stands for itself), and in `calls_at` what `at` was.
struct Recorder {
  PyObject_HEAD
  PyObject *nn, *x, *input, *calls, *calls_at, *at;
};

PyObject *note(Recorder *r, const char *name, const char *spec, PyObject *const *args, Py_ssize_t n)
{
  const Py_ssize_t want = (Py_ssize_t)strlen(spec);  // (what has been left out is zero or null)
  PyObject *a = PyTuple_New(want > n ? want : n);
  if (!a) return nullptr;
  for (Py_ssize_t i = 0; i < PyTuple_GET_SIZE(a); i++) {
    PyObject *o = i >= n ? (spec[i] == 'p' ? Py_None : nullptr) : (i < want && spec[i] == 'p' && args[i] == r->x) ? r->input : args[i];
    if (o) Py_INCREF(o);
    else if (!(o = PyLong_FromLong(0))) {
      Py_DECREF(a);
      return nullptr;
    }
    PyTuple_SET_ITEM(a, i, o);
  }
  PyObject *call = Py_BuildValue("(sN)", name, a);
  const bool ok = call && !PyList_Append(r->calls, call) && !PyList_Append(r->calls_at, r->at);
  Py_XDECREF(call);
  if (!ok) return nullptr;
  Py_RETURN_NONE;
}

template <int F>
PyObject *recorded(PyObject *self, PyObject *const *args, Py_ssize_t n)
{
  Recorder *r = (Recorder *)self;
  PyObject *done = method<F>(r->nn, args, n, nullptr);
  if (!done) return nullptr;
  Py_DECREF(done);
  return note(r, fn_names[F], kinds[fn_kind[F]].spec, args, n);
}

// (the chain is a Python method of nn: it fills the block structs)
PyObject *recorded_chain(PyObject *self, PyObject *const *args, Py_ssize_t n)
{
  Recorder *r = (Recorder *)self;
  PyObject *m = PyObject_GetAttrString(r->nn, "dw_pw_chain_hwc");
  PyObject *done = m ? PyObject_Vectorcall(m, args, (size_t)n, nullptr) : nullptr;
  Py_XDECREF(m);
  if (!done) return nullptr;
  Py_DECREF(done);
  return note(r, fn_names[F_CHAIN], "ppiii", args, n);
}

PyObject *recorder_set_batch(PyObject *self, PyObject *n) { return set_batch(((Recorder *)self)->nn, n); }

PyObject *recorder_new(PyTypeObject *type, PyObject *args, PyObject *)
{
  PyObject *nn, *x;
  if (!PyArg_ParseTuple(args, "O!O", &BaseType, &nn, &x)) return nullptr;
  Recorder *r = (Recorder *)type->tp_alloc(type, 0);
  if (!r) return nullptr;
  Py_INCREF(r->nn = nn);
  Py_INCREF(r->x = x);
  r->calls = PyList_New(0);
  r->calls_at = PyList_New(0);
  Py_INCREF(r->at = Py_None);
  if (PyLong_Check(x)) Py_INCREF(r->input = x);
  else r->input = PyObject_CallNoArgs((PyObject *)&PyBaseObject_Type);
  if (r->calls && r->calls_at && r->input) return (PyObject *)r;
  Py_DECREF(r);
  return nullptr;
}

void recorder_dealloc(PyObject *self)
{
  Recorder *r = (Recorder *)self;
  for (PyObject *o : {r->nn, r->x, r->input, r->calls, r->calls_at, r->at}) Py_XDECREF(o);
  Py_TYPE(self)->tp_free(self);
}

#define R(F, NAME) {NAME, (PyCFunction)(void (*)(void))recorded<F>, METH_FASTCALL, nullptr}
PyMethodDef recorder_methods[] = {
    R(F_CONV_HO, "pulp_nn_conv_Ho_parallel"),
    R(F_PW_HOWO, "pulp_nn_pointwise_HoWo_parallel"),
    R(F_DW_GENERIC, "pulp_nn_depthwise_generic"),
    R(F_LINEAR, "pulp_nn_linear"),
    R(F_LINEAR32, "pulp_nn_linear_out_32"),
    R(F_MAXPOOL, "pulp_nn_maxpool"),
    R(F_AVGPOOL, "pulp_nn_avgpool"),
    R(F_ADD, "pulp_nn_add"),
    R(F_HWC2CHW, "hwc_to_chw"),
    R(F_DWHWC, "depthwise_hwc"),
    R(F_DWPW, "dw_pw_hwc"),
    {"dw_pw_chain_hwc", (PyCFunction)(void (*)(void))recorded_chain, METH_FASTCALL, nullptr},
    {"set_batch", recorder_set_batch, METH_O, nullptr},
    {nullptr, nullptr, 0, nullptr}};
PyMemberDef recorder_members[] = {{"calls", T_OBJECT, offsetof(Recorder, calls), READONLY, nullptr},
                                  {"calls_at", T_OBJECT, offsetof(Recorder, calls_at), READONLY, nullptr},
                                  {"input", T_OBJECT, offsetof(Recorder, input), READONLY, nullptr},
                                  {"at", T_OBJECT, offsetof(Recorder, at), 0, nullptr},
                                  {nullptr, 0, 0, 0, nullptr}};
PyTypeObject RecorderType = {PyVarObject_HEAD_INIT(nullptr, 0)};

// ---- Plan ---------------------------------------------------------------------------------------------------------------

// Addresses are asked for at each run, as a call by itself would: a tensor may have been given other storage since.
struct Call {
  int f;
  Args a;
  PyObject *owner[10];  // what pointer i belongs to; null: the chain's input
  PyObject *blocks;  // the chain entry point's, a tuple
  size_t n_blocks;
};
// what the plan was made from: dict[key] was value (null: absent); items: what a list held, which may change in place
struct Guard {
  PyObject *dict, *key, *value, *items;
};
// a dictionary of which every entry counts, with as many of them as there were (guards of these follow each other)
struct Whole {
  PyObject *dict;
  Py_ssize_t size;
};
struct Plan {
  PyObject_HEAD
  PyObject *nn;      // Base
  PyObject *keep;    // the argument tuples: whatever owns the addresses
  std::vector<Call> *calls;
  std::vector<Guard> *guards;
  std::vector<Whole> *wholes;
  unsigned batch;
};

int fn_index(const char *name)
{
  for (int f = 0; f < F_SET_BATCH; f++)
    if (!strcmp(fn_names[f], name)) return f;
  return -1;
}

bool block_from(PyObject *t, pulp_nn_hip_block *b)
{
  if (!PyTuple_Check(t) || PyTuple_GET_SIZE(t) != 16) {
    PyErr_SetString(PyExc_TypeError, "a block is a tuple of 16");
    return false;
  }
  void *p[8];
  int64_t s[8];
  for (int half = 0, np = 0, ns = 0; half < 2; half++)
    for (int i = 0; i < 8; i++) {
      PyObject *o = PyTuple_GET_ITEM(t, 8 * half + i);
      if (i < 4 ? !to_ptr(o, &p[np++]) : !to_int(o, &s[ns++])) return false;
    }
  *b = pulp_nn_hip_block{(const i8 *)p[0], (const i8 *)p[1], p[2], p[3], (u16)s[0], (u16)s[1], (i8)s[2], (i8)s[3],
                         (const i8 *)p[4], (const i8 *)p[5], p[6], p[7], (u16)s[4], (u16)s[5], (i8)s[6], (i8)s[7]};
  return true;
}

// the same value: the same object, or an equal int
int same(PyObject *a, PyObject *b)
{
  if (a == b) return 1;
  if (!a || !b || !PyLong_CheckExact(a) || !PyLong_CheckExact(b)) return 0;
  return PyObject_RichCompareBool(a, b, Py_EQ);
}

// 1 if the entry is what it was, 0 if not, -1 with an exception set
int unchanged(const Guard &g)
{
  PyObject *v = PyDict_GetItem(g.dict, g.key);
  const int eq = same(v, g.value);
  if (eq != 1 || !g.items) return eq;
  if (PyList_GET_SIZE(v) != PyTuple_GET_SIZE(g.items)) return 0;
  for (Py_ssize_t i = 0; i < PyList_GET_SIZE(v); i++) {
    const int e = same(PyList_GET_ITEM(v, i), PyTuple_GET_ITEM(g.items, i));
    if (e != 1) return e;
  }
  return 1;
}

bool add_guard(Plan *pl, PyObject *dict, PyObject *key, PyObject *value)
{
  Guard g = {dict, key, value, nullptr};
  if (value && PyList_Check(value) && !(g.items = PyList_AsTuple(value))) return false;
  Py_INCREF(g.dict);
  Py_INCREF(g.key);
  Py_XINCREF(g.value);
  pl->guards->push_back(g);
  return true;
}

// a value that cannot change in place, or a list, whose items are kept
bool is_scalar(PyObject *v)
{
  if (PyLong_CheckExact(v)) return true;
  if (v == Py_None || PyLong_Check(v) || PyFloat_Check(v) || PyUnicode_Check(v) || PyTuple_Check(v) || PyList_Check(v)) return true;
  if (!PyNumber_Check(v) || Py_TYPE(v)->tp_hash == PyObject_HashNotImplemented) return false;
  return !PyObject_HasAttrString(v, "data_ptr");  // (numpy's scalars, and no tensor)
}

bool guard_dict(Plan *pl, PyObject *dict, PyObject *which)
{
  PyObject *key, *value;
  if (!PyDict_Check(dict) || (which != Py_None && !PyAnySet_Check(which) && !PyTuple_Check(which))) {
    PyErr_SetString(PyExc_TypeError, "a plan is made from dictionaries, and keys in a tuple, a set or None");
    return false;
  }
  if (PyTuple_Check(which)) {
    for (Py_ssize_t j = 0; j < PyTuple_GET_SIZE(which); j++)
      if (!add_guard(pl, dict, PyTuple_GET_ITEM(which, j), PyDict_GetItem(dict, PyTuple_GET_ITEM(which, j)))) return false;
    return true;
  }
  for (Py_ssize_t pos = 0; PyDict_Next(dict, &pos, &key, &value);) {
    if (!add_guard(pl, dict, key, value)) return false;
    if (which == Py_None || is_scalar(value)) continue;
    const int object = PySet_Contains(which, key);
    if (!object) PyErr_Format(PyExc_TypeError, "%R is a %.100s, which may change in place", key, Py_TYPE(value)->tp_name);
    if (object != 1) return false;
  }
  Py_INCREF(dict);
  pl->wholes->push_back(Whole{dict, PyDict_Size(dict)});
  return true;
}

// Plan(nn, batch, [(entry point, arguments), ...], input, [(dict or list of them, which), ...]): `input` is the object that stands
// for the chain's input in the arguments.  The chain entry point's arguments are (x, out, dim_x, dim_y, ch, [block, ...]).  The
// pairs name the entries the calls were made from, as a tuple of keys, None (all of the dictionary's, and that there are no
// others) or a set (the same; the values of other keys than these have to be numbers, texts, tuples or lists, not arrays, which
// change in place): run() does nothing once one of them has changed, a list's items included.
int plan_init(PyObject *self, PyObject *args, PyObject *)
{
  Plan *pl = (Plan *)self;
  PyObject *nn, *list, *input, *from;
  if (pl->nn) {
    PyErr_SetString(PyExc_RuntimeError, "already initialised");
    return -1;
  }
  if (!PyArg_ParseTuple(args, "O!IO!OO!", &BaseType, &nn, &pl->batch, &PyList_Type, &list, &input, &PyList_Type, &from)) return -1;
  if (!bound((Base *)nn)) return -1;
  Py_INCREF(nn);
  pl->nn = nn;
  Py_INCREF(list);
  pl->keep = list;
  pl->calls = new std::vector<Call>();
  pl->guards = new std::vector<Guard>();
  pl->wholes = new std::vector<Whole>();
  pl->calls->reserve((size_t)PyList_GET_SIZE(list));
  pl->guards->reserve(32 * (size_t)PyList_GET_SIZE(list));
  for (Py_ssize_t i = 0; i < PyList_GET_SIZE(from); i++) {
    PyObject *of, *which;
    if (!PyArg_ParseTuple(PyList_GET_ITEM(from, i), "OO", &of, &which)) return -1;
    if (!PyList_Check(of)) {
      if (!guard_dict(pl, of, which)) return -1;
      continue;
    }
    for (Py_ssize_t j = 0; j < PyList_GET_SIZE(of); j++)
      if (!guard_dict(pl, PyList_GET_ITEM(of, j), which)) return -1;
  }
  for (Py_ssize_t i = 0; i < PyList_GET_SIZE(list); i++) {
    const char *name;
    PyObject *a;
    if (!PyArg_ParseTuple(PyList_GET_ITEM(list, i), "sO!", &name, &PyTuple_Type, &a)) return -1;
    Call c = {};
    c.f = fn_index(name);
    if (c.f < 0) {
      PyErr_Format(PyExc_ValueError, "unknown entry point %s", name);
      return -1;
    }
    std::vector<PyObject *> v;
    const Py_ssize_t n = fn_kind[c.f] == CHAIN ? 5 : PyTuple_GET_SIZE(a);
    const char *spec = fn_kind[c.f] == CHAIN ? "ppiii" : kinds[fn_kind[c.f]].spec;
    if (PyTuple_GET_SIZE(a) < n || (Py_ssize_t)strlen(spec) != n) {
      PyErr_Format(PyExc_ValueError, "wrong number of arguments for %s", name);
      return -1;
    }
    int np = 0, ns = 0;
    for (PyObject *&o : c.owner) o = Py_None;
    for (Py_ssize_t j = 0; j < n; j++) {
      PyObject *o = PyTuple_GET_ITEM(a, j);
      if (spec[j] == 'p') {
        if (o != input && !to_ptr(o, &c.a.p[np])) return -1;
        c.owner[np++] = o == input ? nullptr : o;
      } else if (!to_int(o, &c.a.s[ns++])) {
        return -1;
      }
    }
    if (fn_kind[c.f] == CHAIN) {
      PyObject *list_of = PyTuple_GetItem(a, 5);
      if (!list_of) return -1;
      if (!PyList_Check(list_of)) {
        PyErr_SetString(PyExc_TypeError, "the blocks are a list");
        return -1;
      }
      c.blocks = PyList_AsTuple(list_of);
      if (!c.blocks) return -1;
      c.n_blocks = (size_t)PyTuple_GET_SIZE(c.blocks);
      for (size_t j = 0; j < c.n_blocks; j++) {
        pulp_nn_hip_block b;
        if (block_from(PyTuple_GET_ITEM(c.blocks, j), &b)) continue;
        Py_DECREF(c.blocks);
        return -1;
      }
    }
    pl->calls->push_back(c);
  }
  return 0;
}

// run(x): queues every call with x as the chain's input; raises like the calls themselves would.  False, with nothing
// queued, if what the plan was made from has changed.  Where the library has no kernel for a call on these addresses
// (code 2): the call's index, with the calls in front of it queued and none from it on.
PyObject *plan_run(PyObject *self, PyObject *x)
{
  Plan *pl = (Plan *)self;
  Base *b = (Base *)pl->nn;
  if (!b || !pl->calls) {
    PyErr_SetString(PyExc_RuntimeError, "the plan has not been made");
    return nullptr;
  }
  for (const Whole &w : *pl->wholes)
    if (PyDict_Size(w.dict) != w.size) Py_RETURN_FALSE;
  for (const Guard &g : *pl->guards) {
    const int is = unchanged(g);
    if (is < 0) return nullptr;
    if (!is) Py_RETURN_FALSE;
  }
  // A run's addresses are its own: another thread may enter while this one queues without the interpreter lock.
  std::vector<Args> args;
  std::vector<pulp_nn_hip_block> blocks;
  try {
    args.reserve(pl->calls->size());
    for (const Call &c : *pl->calls) {
      args.push_back(c.a);
      for (int i = 0; i < 10; i++)
        if (c.owner[i] != Py_None && !to_ptr(c.owner[i] ? c.owner[i] : x, &args.back().p[i])) return nullptr;
      for (size_t i = 0; i < c.n_blocks; i++) {
        blocks.emplace_back();
        if (!block_from(PyTuple_GET_ITEM(c.blocks, i), &blocks.back())) return nullptr;
      }
    }
  } catch (const std::bad_alloc &) {
    return PyErr_NoMemory();
  }
  int err = 0;
  size_t j = 0;
  Py_BEGIN_ALLOW_THREADS
  ((void (*)(unsigned))b->fn[F_SET_BATCH])(pl->batch);
  const pulp_nn_hip_block *next = blocks.data();
  for (; j < args.size(); j++) {
    const Call &c = (*pl->calls)[j];
    invoke(b, c.f, args[j], next, (unsigned)c.n_blocks);
    next += c.n_blocks;
    if (b->check && (err = last_error(b))) break;
  }
  Py_END_ALLOW_THREADS
  if (err == PULP_NN_HIP_ERR_UNSUPPORTED) {
    PyObject *r = PyObject_CallMethod(pl->nn, "clear_error", nullptr);
    if (!r) return nullptr;
    Py_DECREF(r);
    return PyLong_FromSize_t(j);
  }
  if (err) return PyObject_CallMethod(pl->nn, "_raise", nullptr);
  Py_RETURN_TRUE;
}

void plan_dealloc(PyObject *self)
{
  Plan *pl = (Plan *)self;
  Py_XDECREF(pl->nn);
  Py_XDECREF(pl->keep);
  if (pl->guards)
    for (Guard &g : *pl->guards) {
      Py_XDECREF(g.dict);
      Py_XDECREF(g.key);
      Py_XDECREF(g.value);
      Py_XDECREF(g.items);
    }
  if (pl->wholes)
    for (Whole &w : *pl->wholes) Py_DECREF(w.dict);
  delete pl->wholes;
  if (pl->calls)
    for (Call &c : *pl->calls) Py_XDECREF(c.blocks);
  delete pl->guards;
  delete pl->calls;
  Py_TYPE(self)->tp_free(self);
}

// plain(nn, {name: attribute}): whether nn is a library object on which every name is found with that attribute, that is, no
// subclass and no attribute of the object itself overrides one.
PyObject *plain(PyObject *, PyObject *const *args, Py_ssize_t n)
{
  if (n != 2 || !PyDict_Check(args[1])) {
    PyErr_SetString(PyExc_TypeError, "plain(object, {name: attribute})");
    return nullptr;
  }
  if (!PyObject_TypeCheck(args[0], &BaseType)) Py_RETURN_FALSE;
  PyObject *key, *value, **own = _PyObject_GetDictPtr(args[0]);
  for (Py_ssize_t pos = 0; PyDict_Next(args[1], &pos, &key, &value);)
    if (_PyType_Lookup(Py_TYPE(args[0]), key) != value) Py_RETURN_FALSE;
  if (own && *own)
    for (Py_ssize_t pos = 0; PyDict_Next(*own, &pos, &key, &value);)
      if (PyDict_GetItem(args[1], key)) Py_RETURN_FALSE;
  Py_RETURN_TRUE;
}

// set_tensor_function(address)
PyObject *set_tensor_function(PyObject *, PyObject *address)
{
  void *p = PyLong_AsVoidPtr(address);
  if (PyErr_Occurred()) return nullptr;
  tensor_address = (int (*)(PyObject *, void **))p;
  Py_RETURN_NONE;
}

PyMethodDef module_methods[] = {{"set_tensor_function", set_tensor_function, METH_O, nullptr},
                                {"plain", (PyCFunction)(void (*)(void))plain, METH_FASTCALL, nullptr}, {nullptr, nullptr, 0, nullptr}};
PyMethodDef plan_methods[] = {{"run", plan_run, METH_O, nullptr}, {nullptr, nullptr, 0, nullptr}};
PyTypeObject PlanType = {PyVarObject_HEAD_INIT(nullptr, 0)};

PyModuleDef module = {PyModuleDef_HEAD_INIT, "_pulpnn_fast", nullptr, -1, module_methods};

}  // namespace

PyMODINIT_FUNC PyInit__pulpnn_fast(void)
{
  BaseType.tp_name = "_pulpnn_fast.Base";
  BaseType.tp_basicsize = sizeof(Base);
  BaseType.tp_flags = Py_TPFLAGS_DEFAULT | Py_TPFLAGS_BASETYPE;
  BaseType.tp_new = PyType_GenericNew;
  BaseType.tp_methods = base_methods;
  BaseType.tp_getset = base_getset;
  PlanType.tp_name = "_pulpnn_fast.Plan";
  PlanType.tp_basicsize = sizeof(Plan);
  PlanType.tp_flags = Py_TPFLAGS_DEFAULT;
  PlanType.tp_new = PyType_GenericNew;
  PlanType.tp_init = plan_init;
  PlanType.tp_dealloc = plan_dealloc;
  PlanType.tp_methods = plan_methods;
  RecorderType.tp_name = "_pulpnn_fast.Recorder";
  RecorderType.tp_basicsize = sizeof(Recorder);
  RecorderType.tp_flags = Py_TPFLAGS_DEFAULT;
  RecorderType.tp_new = recorder_new;
  RecorderType.tp_dealloc = recorder_dealloc;
  RecorderType.tp_methods = recorder_methods;
  RecorderType.tp_members = recorder_members;
  if (PyType_Ready(&BaseType) < 0 || PyType_Ready(&PlanType) < 0 || PyType_Ready(&RecorderType) < 0) return nullptr;
  PyObject *m = PyModule_Create(&module);
  if (!m) return nullptr;
  Py_INCREF(&BaseType);
  PyModule_AddObject(m, "Base", (PyObject *)&BaseType);
  Py_INCREF(&RecorderType);
  PyModule_AddObject(m, "Recorder", (PyObject *)&RecorderType);
  Py_INCREF(&PlanType);
  PyModule_AddObject(m, "Plan", (PyObject *)&PlanType);
  return m;
}
