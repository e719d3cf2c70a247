// Native readers of Python containers of torch tensors: the tables a call hands to libmxplace.so, filled from the
// tensors' C++ objects.  A call over thousands of per-expert tensors, or over every module of a model, spent several
// times its device time in the interpreter asking each for its shape, dtype, layout and address.
//
// Every function is the quick half of a Python function of the same meaning that stands beside its caller: it looks at
// everything that one looks at, on every call, and answers None (or stops early) for whatever is not the plain case - a
// tensor subclass, a tensor without storage or with symbolic sizes, a container or a number of another type, an
// attribute a class defines itself, a check that fails.  The caller then runs the Python half, which decides and words
// the error.  Nothing is kept between calls.
#include <Python.h>
#include <torch/csrc/Dtype.h>
#include <torch/csrc/DynamicTypes.h>
#include <torch/csrc/Exceptions.h>
#include <torch/csrc/autograd/python_variable.h>

#include <cstdint>
#include <cstdio>
#include <cstring>
#include <unordered_map>
#include <unordered_set>
#include <vector>

namespace {

// A reference given up when it goes out of scope.
struct Ref {
  PyObject* p;
  explicit Ref(PyObject* o = nullptr) : p(o) {}
  Ref(const Ref&) = delete;
  Ref& operator=(const Ref&) = delete;
  ~Ref() { Py_XDECREF(p); }
  explicit operator bool() const { return p != nullptr; }
};

// The tensor behind `o`, if it is an ordinary one in memory of its own: exactly Tensor or Parameter, strided, with
// storage (not a functorch wrapper) and sizes that are numbers.
const at::Tensor* plain_tensor(PyObject* o) {
  if (!o || !THPVariable_CheckExact(o)) return nullptr;
  const at::Tensor& t = THPVariable_Unpack(o);
  if (!t.defined() || t.layout() != at::kStrided || !t.has_storage() || t.unsafeGetTensorImpl()->has_symbolic_sizes_strides()) return nullptr;
  return &t;
}

int64_t address(const at::Tensor& t) { return static_cast<int64_t>(reinterpret_cast<intptr_t>(t.data_ptr())); }

bool small_int(PyObject* o, int64_t& out) {
  if (!o || !PyLong_CheckExact(o)) return false;
  int overflow = 0;
  out = PyLong_AsLongLongAndOverflow(o, &overflow);
  return overflow == 0;
}

// The numbers of a tuple (torch.Size among them) or list of at most `cap`; -1 for anything else.
int dims_of(PyObject* seq, int64_t* out, int cap) {
  const bool tuple = PyTuple_Check(seq);
  if (!tuple && !PyList_CheckExact(seq)) return -1;
  const Py_ssize_t n = tuple ? PyTuple_GET_SIZE(seq) : PyList_GET_SIZE(seq);
  if (n > cap) return -1;
  for (Py_ssize_t k = 0; k < n; ++k)
    if (!small_int(tuple ? PyTuple_GET_ITEM(seq, k) : PyList_GET_ITEM(seq, k), out[k])) return -1;
  return (int)n;
}

PyObject* interned(const char* s) { return PyUnicode_InternFromString(s); }

struct Names {
  PyObject *src = interned("src"), *dst = interned("dst"), *shape = interned("shape"), *elem_size = interned("elem_size"),
           *cast = interned("cast"), *src_strides = interned("src_strides"), *dst_strides = interned("dst_strides");
  PyObject *modules = interned("_modules"), *parameters = interned("_parameters"), *buffers = interned("_buffers");
  PyObject *named_modules = interned("named_modules"), *getattr = interned("__getattr__"), *getattribute = interned("__getattribute__");
  PyObject *kv_b_proj = interned("kv_b_proj"), *weight = interned("weight"), *w_uv = interned("W_UV"), *w_uk_t = interned("W_UK_T"),
           *num_heads = interned("num_heads"), *nope = interned("qk_nope_head_dim"), *v_dim = interned("v_head_dim");
  PyObject *name = interned("name"), *dtype = interned("dtype"), *nbytes = interned("nbytes"), *checksum = interned("checksum"),
           *digest = interned("digest");
};
Names* N = nullptr;

// The 28 words of a mxp_view_copy: src, dst, ndim | elem_size << 32, cast | contiguous flags << 32, shape, source strides,
// destination strides.
constexpr int kViewWords = 28, kMaxDims = 8;

// addresses(held, meta, contiguous): the address of the tensor held under every name of `meta` ({name: (shape, dtype)}), as
// native 64-bit words, when each has that shape and dtype (and is contiguous, if asked).
PyObject* addresses(PyObject*, PyObject* args) {
  HANDLE_TH_ERRORS
  PyObject *held, *meta;
  int contiguous;
  if (!PyArg_ParseTuple(args, "OOp", &held, &meta, &contiguous)) return nullptr;
  if (!PyDict_CheckExact(held) || !PyDict_CheckExact(meta)) Py_RETURN_NONE;
  std::vector<int64_t> out;
  out.reserve((size_t)PyDict_GET_SIZE(meta));
  PyObject *key, *value;
  Py_ssize_t pos = 0;
  while (PyDict_Next(meta, &pos, &key, &value)) {
    if (!PyUnicode_CheckExact(key) || !PyTuple_CheckExact(value) || PyTuple_GET_SIZE(value) != 2) Py_RETURN_NONE;
    const at::Tensor* t = plain_tensor(PyDict_GetItemWithError(held, key));
    if (!t) {
      PyErr_Clear();
      Py_RETURN_NONE;
    }
    PyObject* shape = PyTuple_GET_ITEM(value, 0);
    const auto sizes = t->sizes();
    if (!PyTuple_Check(shape) || (size_t)PyTuple_GET_SIZE(shape) != sizes.size()) Py_RETURN_NONE;
    for (size_t d = 0; d < sizes.size(); ++d) {
      int64_t n;
      if (!small_int(PyTuple_GET_ITEM(shape, (Py_ssize_t)d), n) || n != sizes[d]) Py_RETURN_NONE;
    }
    if (reinterpret_cast<PyObject*>(torch::getTHPDtype(t->scalar_type())) != PyTuple_GET_ITEM(value, 1)) Py_RETURN_NONE;
    if (contiguous && !t->is_contiguous()) Py_RETURN_NONE;
    out.push_back(address(*t));
  }
  return PyBytes_FromStringAndSize(reinterpret_cast<const char*>(out.data()), (Py_ssize_t)(out.size() * sizeof(int64_t)));
  END_HANDLE_TH_ERRORS
}

// pointers(buffers): the address of every tensor, or the number, of a list or tuple, as native 64-bit words.
PyObject* pointers(PyObject*, PyObject* seq) {
  HANDLE_TH_ERRORS
  const bool tuple = PyTuple_CheckExact(seq);
  if (!tuple && !PyList_CheckExact(seq)) Py_RETURN_NONE;
  const Py_ssize_t n = tuple ? PyTuple_GET_SIZE(seq) : PyList_GET_SIZE(seq);
  std::vector<int64_t> out((size_t)n);
  for (Py_ssize_t k = 0; k < n; ++k) {
    PyObject* o = tuple ? PyTuple_GET_ITEM(seq, k) : PyList_GET_ITEM(seq, k);
    if (const at::Tensor* t = plain_tensor(o)) out[(size_t)k] = address(*t);
    else if (!small_int(o, out[(size_t)k]) || out[(size_t)k] < 0) Py_RETURN_NONE;
  }
  return PyBytes_FromStringAndSize(reinterpret_cast<const char*>(out.data()), n * (Py_ssize_t)sizeof(int64_t));
  END_HANDLE_TH_ERRORS
}

bool put_view(PyObject* v, int64_t* w) {
  if (!PyDict_CheckExact(v)) return false;
  auto item = [&](PyObject* key) { return PyDict_GetItemWithError(v, key); };
  auto place = [&](PyObject* o, int64_t& at) {
    if (const at::Tensor* t = plain_tensor(o)) {
      at = address(*t);
      return true;
    }
    return small_int(o, at);
  };
  int64_t elem = 0, cast = 0;
  PyObject *shape = item(N->shape), *ss = item(N->src_strides), *ds = item(N->dst_strides), *c = item(N->cast);
  if (!shape || !place(item(N->src), w[0]) || !place(item(N->dst), w[1]) || !small_int(item(N->elem_size), elem)) return false;
  if (c && !small_int(c, cast)) return false;
  if (elem < 0 || elem > INT32_MAX || cast < 0 || cast > INT32_MAX) return false;
  const bool no_ss = !ss || ss == Py_None, no_ds = !ds || ds == Py_None;
  const int nd = dims_of(shape, w + 4, kMaxDims);
  if (nd < 0 || (!no_ss && dims_of(ss, w + 12, kMaxDims) < 0) || (!no_ds && dims_of(ds, w + 20, kMaxDims) < 0)) return false;
  w[2] = (int64_t)nd | elem << 32;
  w[3] = cast | (int64_t)no_ss << 32 | (int64_t)no_ds << 40;
  return true;
}

// put_views(views, words, first): fills the words of views first, first + 1, ... of a list or tuple of dicts; returns the
// index of the first one it leaves alone (its words zero), or their number.
PyObject* put_views(PyObject*, PyObject* args) {
  HANDLE_TH_ERRORS
  PyObject *views, *words;
  Py_ssize_t first;
  if (!PyArg_ParseTuple(args, "OOn", &views, &words, &first)) return nullptr;
  const bool tuple = PyTuple_CheckExact(views);
  if (first < 0 || (!tuple && !PyList_CheckExact(views))) return PyLong_FromSsize_t(first);
  Py_buffer buf;
  if (PyObject_GetBuffer(words, &buf, PyBUF_WRITABLE) != 0) return nullptr;
  const Py_ssize_t n = tuple ? PyTuple_GET_SIZE(views) : PyList_GET_SIZE(views);
  Py_ssize_t k = first;
  try {
    for (; k < n && (k + 1) * kViewWords * (Py_ssize_t)sizeof(int64_t) <= buf.len; ++k) {
      int64_t* w = static_cast<int64_t*>(buf.buf) + k * kViewWords;
      if (put_view(tuple ? PyTuple_GET_ITEM(views, k) : PyList_GET_ITEM(views, k), w)) continue;
      std::memset(w, 0, kViewWords * sizeof(int64_t));
      break;
    }
  } catch (...) {
    PyBuffer_Release(&buf);
    throw;
  }
  PyBuffer_Release(&buf);
  PyErr_Clear();
  return PyLong_FromSsize_t(k);
  END_HANDLE_TH_ERRORS
}

// ---- modules ---------------------------------------------------------------------------------------------------------
// Attribute lookup of torch.nn.Module without its __getattr__, for classes that leave the lookup as it is.
struct ModuleReader {
  enum Use { kNothing, kWalk, kRead };
  PyObject* base;  // torch.nn.Module
  Ref named_modules, getattr;
  std::unordered_map<PyTypeObject*, Use> usable;
  explicit ModuleReader(PyObject* module_class)
      : base(module_class), named_modules(PyObject_GetAttr(module_class, N->named_modules)), getattr(PyObject_GetAttr(module_class, N->getattr)) {}

  // What can be done with instances of the type.  Walked: a Module whose walk and identity are Module's.  Read: one whose
  // attribute lookup is Module's as well, with none of the attributes we ask for defined by the class.
  Use use(PyObject* o) {
    PyTypeObject* type = Py_TYPE(o);
    const auto found = usable.find(type);
    if (found != usable.end()) return found->second;
    Use u = PyType_IsSubtype(type, reinterpret_cast<PyTypeObject*>(base)) && type->tp_hash == PyBaseObject_Type.tp_hash &&
                    _PyType_Lookup(type, N->named_modules) == named_modules.p && !_PyType_Lookup(type, N->modules) &&
                    _PyType_Lookup(type, N->getattribute) == _PyType_Lookup(&PyBaseObject_Type, N->getattribute)
                ? kRead
                : kNothing;
    if (u == kRead && _PyType_Lookup(type, N->getattr) != getattr.p) u = kWalk;
    for (PyObject* name : {N->kv_b_proj, N->weight, N->w_uv, N->w_uk_t, N->num_heads, N->nope, N->v_dim, N->parameters, N->buffers})
      if (u == kRead && _PyType_Lookup(type, name)) u = kWalk;
    usable.emplace(type, u);
    return u;
  }
  bool can_read(PyObject* o) { return use(o) == kRead; }
  // Borrowed; null if the attribute is absent.  `ok` turns false where the instance is not laid out as expected.
  PyObject* get(PyObject* dict, PyObject* name, bool& ok) {
    if (PyObject* v = PyDict_GetItemWithError(dict, name)) return v;
    for (PyObject* group : {N->parameters, N->buffers, N->modules}) {
      PyObject* g = PyDict_GetItemWithError(dict, group);
      if (!g || !PyDict_CheckExact(g)) {
        ok = false;
        return nullptr;
      }
      if (PyObject* v = PyDict_GetItemWithError(g, name)) return v;
    }
    return nullptr;
  }
};

// MXP_CAST_* for a pair of element types; -1 where there is no entry.
int cast_code(at::ScalarType s, at::ScalarType d) {
  using T = at::ScalarType;
  if (s != T::Float && s != T::BFloat16 && s != T::Half && s != T::Float8_e4m3fn) return -1;
  if (s == d) return 0;
  if (s == T::Float && d == T::BFloat16) return 1;
  if (s == T::BFloat16 && d == T::Float) return 2;
  if (s == T::Half && d == T::Float) return 3;
  if (s == T::Float && d == T::Half) return 4;
  if (s == T::Float8_e4m3fn && d == T::BFloat16) return 5;
  if (s == T::Half && d == T::BFloat16) return 6;
  if (s == T::BFloat16 && d == T::Half) return 7;
  return -1;
}

struct MlaWalk {
  ModuleReader read;
  PyObject* general;  // the Python function for one module, or null
  bool raised = false;
  std::unordered_set<PyObject*> seen;
  std::vector<int64_t> words;
  MlaWalk(PyObject* module_class, PyObject* for_one_module) : read(module_class), general(for_one_module) {}

  bool visit(PyObject* m, int depth) {
    if (depth > 200) return false;
    const ModuleReader::Use use = read.use(m);
    if (use == ModuleReader::kNothing || (use == ModuleReader::kWalk && !general)) return false;
    if (!seen.insert(m).second) return true;
    Ref dict(PyObject_GenericGetDict(m, nullptr));
    if (!dict) return false;
    bool done = use == ModuleReader::kRead;
    if (done) {
      const size_t before = words.size();
      PyObject* proj = read.get(dict.p, N->kv_b_proj, done);
      done = done && (!proj || views_of(dict.p, proj));
      if (!done) words.resize(before);
    }
    if (!done && !ask(m)) return false;
    PyObject* modules = PyDict_GetItemWithError(dict.p, N->modules);
    if (!modules || !PyDict_CheckExact(modules)) return false;
    if (PyDict_GET_SIZE(modules) == 0) return true;
    const Ref children(PyDict_Values(modules));  // of their own: asking may run any code
    if (!children) return false;
    for (Py_ssize_t k = 0; k < PyList_GET_SIZE(children.p); ++k) {
      PyObject* child = PyList_GET_ITEM(children.p, k);
      if (child != Py_None && !visit(child, depth + 1)) return false;
    }
    return true;
  }

  // The views of a module that is not the plain case, by the Python function.
  bool ask(PyObject* m) {
    if (!general) return false;
    PyErr_Clear();
    const Ref got(PyObject_CallFunctionObjArgs(general, m, nullptr));
    Py_buffer buf;
    if (!got || PyObject_GetBuffer(got.p, &buf, PyBUF_SIMPLE) != 0) {
      raised = true;
      return false;
    }
    const size_t before = words.size(), n = (size_t)buf.len / sizeof(int64_t);
    words.resize(before + n);
    std::memcpy(words.data() + before, buf.buf, n * sizeof(int64_t));
    PyBuffer_Release(&buf);
    return true;
  }

  bool views_of(PyObject* dict, PyObject* proj) {
    bool ok = true;
    PyObject* const outs[2] = {read.get(dict, N->w_uv, ok), read.get(dict, N->w_uk_t, ok)};
    if (!ok) return false;
    if (!outs[0] && !outs[1]) return true;  // no absorbed weights
    if (proj == Py_None || !read.can_read(proj)) return false;
    Ref proj_dict(PyObject_GenericGetDict(proj, nullptr));
    if (!proj_dict) return false;
    const at::Tensor* w = plain_tensor(read.get(proj_dict.p, N->weight, ok));
    int64_t heads, nope, v_dim;
    if (!w || !ok || !small_int(read.get(dict, N->num_heads, ok), heads) || !small_int(read.get(dict, N->nope, ok), nope) ||
        !small_int(read.get(dict, N->v_dim, ok), v_dim))
      return false;
    const int64_t limit = 1 << 24;
    if (heads < 0 || nope < 0 || v_dim < 0 || heads > limit || nope > limit || v_dim > limit) return false;
    if (w->dim() != 2 || !w->is_contiguous() || w->size(0) != heads * (nope + v_dim)) return false;
    const int64_t latent = w->size(1), head_stride = (nope + v_dim) * latent, es = (int64_t)w->element_size(), src = address(*w);
    const int64_t shapes[2][3] = {{v_dim, heads, latent}, {nope, latent, heads}};
    const int64_t strides[2][3] = {{latent, head_stride, 1}, {latent, 1, head_stride}};
    const int64_t first[2] = {nope * latent, 0};
    for (int k = 0; k < 2; ++k) {
      if (!outs[k] || outs[k] == Py_None) continue;
      const at::Tensor* out = plain_tensor(outs[k]);
      if (!out || out->dim() != 3) return false;
      const int cast = cast_code(w->scalar_type(), out->scalar_type());
      if (cast < 0) return false;
      const size_t at = words.size();
      words.resize(at + kViewWords, 0);
      int64_t* o = words.data() + at;
      o[0] = src + first[k] * es;
      o[1] = address(*out);
      o[2] = 3 | (int64_t)out->element_size() << 32;
      o[3] = cast;
      for (int d = 0; d < 3; ++d) {
        if (out->size(d) != shapes[k][d]) return false;
        o[4 + d] = shapes[k][d];
        o[12 + d] = strides[k][d];
        o[20 + d] = out->stride(d);
      }
    }
    return true;
  }
};

// mla_views(model, module_class[, general]): the views that rewrite W_UV and W_UK_T of every module of the model, in the
// order of named_modules, as a bytearray of mxp_view_copy records.  `general(module)` gives the records of a module that is
// not the plain case, and raises where there are none to give.
PyObject* mla_views(PyObject*, PyObject* args) {
  HANDLE_TH_ERRORS
  PyObject *model, *module_class, *general = nullptr;
  if (!PyArg_ParseTuple(args, "OO|O", &model, &module_class, &general)) return nullptr;
  if (!PyType_Check(module_class)) Py_RETURN_NONE;
  MlaWalk walk(module_class, general);
  if (!walk.read.named_modules || !walk.read.getattr || !walk.visit(model, 0)) {
    if (walk.raised) return nullptr;
    PyErr_Clear();
    Py_RETURN_NONE;
  }
  return PyByteArray_FromStringAndSize(reinterpret_cast<const char*>(walk.words.data()), (Py_ssize_t)(walk.words.size() * sizeof(int64_t)));
  END_HANDLE_TH_ERRORS
}

// state_key(tensors): address, element type, shape and strides of every tensor of a dict in its order, as one bytes object;
// floating-point tensors only.
PyObject* state_key(PyObject*, PyObject* tensors) {
  HANDLE_TH_ERRORS
  if (!PyDict_CheckExact(tensors)) Py_RETURN_NONE;
  std::vector<int64_t> out;
  out.reserve(8 * (size_t)PyDict_GET_SIZE(tensors));
  PyObject *key, *value;
  Py_ssize_t pos = 0;
  while (PyDict_Next(tensors, &pos, &key, &value)) {
    const at::Tensor* t = plain_tensor(value);
    if (!t || !at::isFloatingType(t->scalar_type())) Py_RETURN_NONE;
    out.push_back(address(*t));
    out.push_back((int64_t)t->scalar_type() | (int64_t)t->dim() << 32);
    out.insert(out.end(), t->sizes().begin(), t->sizes().end());
    out.insert(out.end(), t->strides().begin(), t->strides().end());
  }
  return PyBytes_FromStringAndSize(reinterpret_cast<const char*>(out.data()), (Py_ssize_t)(out.size() * sizeof(int64_t)));
  END_HANDLE_TH_ERRORS
}

// param_nbytes(params, spec_class, dtype_sizes): the byte size of every parameter; computed here for instances of
// spec_class with a shape of plain numbers, asked of the object otherwise.  Attributes may run any code, also code that
// changes the list: it is walked as a list iterator walks it, with a reference to the element in hand.
PyObject* param_nbytes(PyObject*, PyObject* args) {
  HANDLE_TH_ERRORS
  PyObject *params, *spec, *sizes;
  if (!PyArg_ParseTuple(args, "OOO!", &params, &spec, &PyDict_Type, &sizes)) return nullptr;
  Ref seq(PySequence_Fast(params, "params must be a sequence"));
  if (!seq) return nullptr;
  Ref out(PyList_New(0));
  if (!out) return nullptr;
  for (Py_ssize_t k = 0; k < PySequence_Fast_GET_SIZE(seq.p); ++k) {
    const Ref p(Py_NewRef(PySequence_Fast_GET_ITEM(seq.p, k)));
    PyObject* value = nullptr;
    if (reinterpret_cast<PyObject*>(Py_TYPE(p.p)) == spec) {
      Ref dict(PyObject_GenericGetDict(p.p, nullptr));
      PyObject* dtype = dict ? PyDict_GetItemWithError(dict.p, N->dtype) : nullptr;
      PyObject* shape = dict ? PyDict_GetItemWithError(dict.p, N->shape) : nullptr;
      int64_t total = 0, dims[32];
      const int nd = shape && PyTuple_Check(shape) ? dims_of(shape, dims, 32) : -1;
      if (dtype && PyUnicode_CheckExact(dtype) && nd >= 0 && small_int(PyDict_GetItemWithError(sizes, dtype), total)) {
        bool fits = true;
        for (int d = 0; d < nd; ++d) fits = fits && !__builtin_mul_overflow(total, dims[d], &total);
        if (fits) value = PyLong_FromLongLong(total);
      }
      PyErr_Clear();
    }
    const Ref size(value ? value : PyObject_GetAttr(p.p, N->nbytes));
    if (!size || PyList_Append(out.p, size.p) != 0) return nullptr;
  }
  Py_INCREF(out.p);
  return out.p;
  END_HANDLE_TH_ERRORS
}

// records(cls, params, nbytes, checksums, digests): an instance of the (frozen) dataclass for each parameter, its fields set
// as its __init__ would leave them.
PyObject* records(PyObject*, PyObject* args) {
  HANDLE_TH_ERRORS
  PyObject *cls, *in[4];
  if (!PyArg_ParseTuple(args, "O!OOOO", &PyType_Type, &cls, &in[0], &in[1], &in[2], &in[3])) return nullptr;
  Ref p(PySequence_Fast(in[0], "params must be a sequence")), nb(PySequence_Fast(in[1], "sizes")), cs(PySequence_Fast(in[2], "checksums")),
      dg(PySequence_Fast(in[3], "digests"));
  if (!p || !nb || !cs || !dg) return nullptr;
  const auto there = [&](Py_ssize_t k) {  // ends with the shortest, as zip() does
    for (PyObject* s : {p.p, nb.p, cs.p, dg.p})
      if (k >= PySequence_Fast_GET_SIZE(s)) return false;
    return true;
  };
  PyTypeObject* type = reinterpret_cast<PyTypeObject*>(cls);
  Ref none(PyTuple_New(0)), out(PyList_New(0));
  if (!none || !out) return nullptr;
  for (Py_ssize_t k = 0; there(k); ++k) {
    const Ref param(Py_NewRef(PySequence_Fast_GET_ITEM(p.p, k))), size(Py_NewRef(PySequence_Fast_GET_ITEM(nb.p, k))),
        sum(Py_NewRef(PySequence_Fast_GET_ITEM(cs.p, k))), digest(Py_NewRef(PySequence_Fast_GET_ITEM(dg.p, k)));
    const Ref name(PyObject_GetAttr(param.p, N->name)), dtype(PyObject_GetAttr(param.p, N->dtype));
    if (!name || !dtype) return nullptr;
    const Ref r(PyBaseObject_Type.tp_new(type, none.p, nullptr));
    if (!r || PyList_Append(out.p, r.p) != 0) return nullptr;
    const Ref dict(PyObject_GenericGetDict(r.p, nullptr));
    if (!dict || PyDict_SetItem(dict.p, N->name, name.p) || PyDict_SetItem(dict.p, N->nbytes, size.p) ||
        PyDict_SetItem(dict.p, N->dtype, dtype.p) || PyDict_SetItem(dict.p, N->checksum, sum.p) || PyDict_SetItem(dict.p, N->digest, digest.p))
      return nullptr;
  }
  Py_INCREF(out.p);
  return out.p;
  END_HANDLE_TH_ERRORS
}

PyMethodDef methods[] = {{"addresses", addresses, METH_VARARGS, nullptr},       {"pointers", pointers, METH_O, nullptr},
                         {"put_views", put_views, METH_VARARGS, nullptr},       {"mla_views", mla_views, METH_VARARGS, nullptr},
                         {"state_key", state_key, METH_O, nullptr},             {"param_nbytes", param_nbytes, METH_VARARGS, nullptr},
                         {"records", records, METH_VARARGS, nullptr},           {nullptr, nullptr, 0, nullptr}};
PyModuleDef module = {PyModuleDef_HEAD_INIT, "_tensors", "Native readers of containers of torch tensors.", -1, methods, nullptr, nullptr, nullptr, nullptr};

}  // namespace

// `built_for`: the interpreter and torch it was compiled against (_lib.tensors_tag), which the caller compares with what it runs in.
PyMODINIT_FUNC PyInit__tensors(void) {
  int major = 0, minor = 0;
  std::sscanf(Py_GetVersion(), "%d.%d", &major, &minor);
  if (major != PY_MAJOR_VERSION || minor != PY_MINOR_VERSION) {  // which lays its objects out differently
    PyErr_SetString(PyExc_ImportError, "built for Python " PY_VERSION);
    return nullptr;
  }
  if (!N) N = new Names();
  PyObject* m = PyModule_Create(&module);
  if (m && PyModule_AddStringConstant(m, "built_for", MXP_BUILT_FOR) != 0) {
    Py_DECREF(m);
    return nullptr;
  }
  return m;
}
