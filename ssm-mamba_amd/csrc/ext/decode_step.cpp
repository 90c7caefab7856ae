// PyTorch-ROCm extension module `decode_step`: the host work of a decode step
// over the C ABI of libssm_mamba_hip.so, for models built from the package's
// own layer classes.
//
//   layer_rows(layers, x, classes) -> bytes | None
//       the SSM_LAYER_* addresses of every Block in `layers`, when
//       decode.layers_supported allows the one-launch step;
//   block_step(block, x, classes, fold, rows) -> Tensor | None
//       Block.step: the fused kernels of one layer, by batch size the GEMV
//       kernels (up to 8 rows) or, with rows, the matrix-core ones (9 to 64).
//
// A step of a 24-layer model reads 14 tensors a layer through nn.Module's
// __getattr__ and checks a dozen properties of each: 600 us a step in Python,
// more than its kernels take (380), and 40 of a single layer's 55.  Measured
// with the checks in Python and here: 24 layers of 1024 at batch 4, 991 us a
// step and 428; one layer at 32 rows, 61 and 30; one of 384 at 2 rows, 55 and
// 15; 12 layers of 128 at 16 rows, 725 and 222.  Here the reads are dictionary
// lookups.  The answer is a whole yes only: the objects must be exactly the
// classes given (no subclass, no attribute of the class in a parameter's
// place), the tensors exactly torch.Tensor or Parameter with storage, and
// every condition of the Python checks must hold.  None leaves the decision to
// those checks, which take any object with the same attributes.  Nothing is
// kept from call to call.
#include "ext_common.h"

#include <torch/csrc/autograd/python_variable.h>
#include <c10/core/impl/TorchDispatchModeTLS.h>

#include <cstring>
#include <initializer_list>

namespace {

using namespace ssm_ext;
namespace py = pybind11;

// ---------------------------------------------------------------- attributes

#define SSM_NAMES(X)                                                                            \
  X(_parameters) X(_buffers) X(_modules) X(_forward_hooks) X(_forward_pre_hooks) X(norm) X(ssm) \
  X(weight) X(bias) X(eps) X(input_proj) X(conv) X(ssm_param_proj) X(delta_proj) X(out_proj)     \
  X(log_A) X(D) X(_conv_context) X(_ssm_hiddens) X(inner_dim) X(state_dim) X(delta_rank)         \
  X(conv_kernel) X(forward) X(step)

struct Names {
#define SSM_DECL(n) PyObject* n = PyUnicode_InternFromString(#n);
  SSM_NAMES(SSM_DECL)
#undef SSM_DECL
};

const Names& names() {
  static const Names* n = new Names();
  return *n;
}

// An nn.Module whose class is exactly cls: its own attributes by the order of
// the normal lookup (the instance's dictionary, then nn.Module.__getattr__'s
// three).  All references are borrowed: the module keeps them.
struct Module {
  PyTypeObject* type = nullptr;
  PyObject* dicts[4] = {};

  bool open(PyObject* o, PyObject* cls) {
    if (!o || reinterpret_cast<PyObject*>(Py_TYPE(o)) != cls) return false;
    type = Py_TYPE(o);
    PyObject** d = _PyObject_GetDictPtr(o);
    if (!d || !*d) return false;
    dicts[0] = *d;
    PyObject* const keys[3] = {names()._parameters, names()._buffers, names()._modules};
    for (int i = 0; i < 3; ++i) {
      dicts[i + 1] = PyDict_GetItem(dicts[0], keys[i]);
      if (!dicts[i + 1] || !PyDict_Check(dicts[i + 1])) return false;
    }
    return true;
  }
  PyObject* get(PyObject* name) const {
    if (_PyType_Lookup(type, name)) return nullptr;
    for (PyObject* d : dicts)
      if (PyObject* v = PyDict_GetItem(d, name)) return v;
    return nullptr;
  }
  bool integer(PyObject* name, int64_t& v) const {
    PyObject* o = get(name);
    if (!o || !PyLong_CheckExact(o)) return false;
    v = PyLong_AsLongLong(o);
    if (v == -1 && PyErr_Occurred()) {
      PyErr_Clear();
      return false;
    }
    return true;
  }
  // a call is the class's forward: none set on the object, no hooks of its own
  bool plain_call() const {
    if (PyDict_GetItem(dicts[0], names().forward)) return false;
    for (PyObject* n : {names()._forward_hooks, names()._forward_pre_hooks}) {
      PyObject* h = PyDict_GetItem(dicts[0], n);
      if (!h || PyObject_Size(h) != 0) return false;
    }
    return true;
  }
};

// The tensor o holds (nullptr: none there, or one with semantics of its own).
const at::Tensor* tensor(PyObject* o) {
  if (!o || !THPVariable_CheckExact(o)) return nullptr;
  const at::Tensor& t = THPVariable_Unpack(o);
  return t.defined() && t.layout() == at::kStrided && t.has_storage() ? &t : nullptr;
}

bool aligned16(const at::Tensor& t) { return (reinterpret_cast<uintptr_t>(t.data_ptr()) & 15) == 0; }

struct Classes {
  PyObject *block, *mamba, *norm, *linear, *conv, *list;
  explicit Classes(const py::tuple& c)
      : block(c[0].ptr()), mamba(c[1].ptr()), norm(c[2].ptr()), linear(c[3].ptr()),
        conv(c[4].ptr()), list(c[5].ptr()) {}
};

// ---------------------------------------------------------------- one layer

struct Step {  // the token batch
  const at::Tensor* x;
  int64_t batch, k;
  int e;  // elements in 16 bytes
  int dtype;

  bool open(PyObject* o, int64_t lo, int64_t hi) {
    if (at::GradMode::is_enabled() || c10::impl::TorchDispatchModeTLS::any_modes_set()) return false;
    x = tensor(o);
    if (!x || !x->is_cuda() || x->dim() != 2) return false;
    const auto t = x->scalar_type();
    if (t != at::kFloat && t != at::kBFloat16) return false;
    dtype = t == at::kBFloat16 ? SSM_BF16 : SSM_F32;
    e = dtype == SSM_BF16 ? 8 : 4;
    batch = x->size(0);
    k = x->size(1);
    return batch >= lo && batch <= hi && k > 0 && k % e == 0 && x->is_contiguous() && aligned16(*x);
  }
  bool fits(const at::Tensor& t) const {
    return t.scalar_type() == x->scalar_type() && t.is_contiguous() && t.device() == x->device() &&
           aligned16(t);
  }
};

struct Layer {
  int64_t dim, nstate, rank, width, nout;
  double eps;
  bool calls_plain;               // norm() and ssm.step() are their classes' own
  void* row[SSM_LAYER_NPTR];

  bool put(const Step& s, int slot, PyObject* o, std::initializer_list<int64_t> shape, bool optional) {
    row[slot] = nullptr;
    if (!o) return false;
    if (o == Py_None) return optional;
    const at::Tensor* t = tensor(o);
    if (!t || !s.fits(*t) || t->sizes() != at::IntArrayRef(shape)) return false;
    row[slot] = t->data_ptr();
    return row[slot] != nullptr;
  }
  bool proj(const Step& s, const Module& ssm, PyObject* name, PyObject* cls, int w_slot, int b_slot,
            std::initializer_list<int64_t> shape) {
    Module m;
    if (!m.open(ssm.get(name), cls)) return false;
    if (!put(s, w_slot, m.get(names().weight), shape, false)) return false;
    PyObject* b = m.get(names().bias);
    return b_slot < 0 ? b == Py_None : put(s, b_slot, b, {*shape.begin()}, true);
  }
  bool cache(const Step& s, int slot, PyObject* o, at::ScalarType type, std::initializer_list<int64_t> shape,
             bool align) {
    const at::Tensor* t = tensor(o);
    if (!t || t->scalar_type() != type || !t->is_contiguous() || t->device() != s.x->device() ||
        t->sizes() != at::IntArrayRef(shape) || (align && !aligned16(*t)))
      return false;
    row[slot] = t->data_ptr();
    return row[slot] != nullptr;
  }

  // Block `o` for the batch s: every condition of decode.block_step_supported
  // (or, past 8 rows, rows_step_supported), and all shapes.
  bool open(const Step& s, PyObject* o, const Classes& c) {
    const Names& n = names();
    Module blk, ssm, norm;
    if (!blk.open(o, c.block) || !ssm.open(blk.get(n.ssm), c.mamba) ||
        !norm.open(blk.get(n.norm), c.norm))
      return false;
    PyObject* ep = norm.get(n.eps);
    if (!ep || !PyFloat_CheckExact(ep)) return false;
    eps = PyFloat_AS_DOUBLE(ep);
    calls_plain = norm.plain_call() && !PyDict_GetItem(ssm.dicts[0], n.step);
    if (!ssm.integer(n.inner_dim, dim) || !ssm.integer(n.state_dim, nstate) ||
        !ssm.integer(n.delta_rank, rank) || !ssm.integer(n.conv_kernel, width))
      return false;
    if (nstate != 4 && nstate != 8 && nstate != 16 && nstate != 32 && nstate != 64) return false;
    if (width < 2 || width > 8 || rank < 1 || dim < 1 || dim % s.e) return false;
    nout = rank + 2 * nstate;
    if (nout > 16384) return false;
    return proj(s, ssm, n.input_proj, c.linear, SSM_LAYER_IN_PROJ_W, SSM_LAYER_IN_PROJ_B,
                {2 * dim, s.k}) &&
           put(s, SSM_LAYER_NORM_W, norm.get(n.weight), {s.k}, false) &&
           proj(s, ssm, n.conv, c.conv, SSM_LAYER_CONV_W, SSM_LAYER_CONV_B, {dim, 1, width}) &&
           proj(s, ssm, n.ssm_param_proj, c.linear, SSM_LAYER_X_PROJ_W, -1, {nout, dim}) &&
           proj(s, ssm, n.delta_proj, c.linear, SSM_LAYER_DT_PROJ_W, SSM_LAYER_DT_BIAS, {dim, rank}) &&
           put(s, SSM_LAYER_LOG_A, ssm.get(n.log_A), {dim, nstate}, false) &&
           put(s, SSM_LAYER_D, ssm.get(n.D), {dim}, true) &&
           proj(s, ssm, n.out_proj, c.linear, SSM_LAYER_OUT_PROJ_W, SSM_LAYER_OUT_PROJ_B, {s.k, dim}) &&
           cache(s, SSM_LAYER_CONV_WINDOW, ssm.get(n._conv_context), s.x->scalar_type(),
                 {s.batch, dim, width - 1}, false) &&
           cache(s, SSM_LAYER_STATE, ssm.get(n._ssm_hiddens), at::kFloat, {s.batch, dim, nstate}, true);
  }
};

// ---------------------------------------------------------------- entries

py::object layer_rows(const py::object& layers, const py::object& x, const py::tuple& classes) {
  const Classes c(classes);
  Step s;
  Module list;
  if (!s.open(x.ptr(), 1, 4) || !list.open(layers.ptr(), c.list)) return py::none();
  PyObject* mods = list.dicts[3];
  const Py_ssize_t count = PyDict_Size(mods);
  if (count < 1) return py::none();
  py::bytes out(nullptr, (size_t)count * SSM_LAYER_NPTR * sizeof(void*));
  char* dst = PyBytes_AS_STRING(out.ptr());
  Layer l, l0;
  Py_ssize_t pos = 0, i = 0;
  PyObject *key, *value;
  while (PyDict_Next(mods, &pos, &key, &value)) {
    if (i >= count || !l.open(s, value, c)) return py::none();
    if (i == 0) {
      l0 = l;
      // decode.layers_supported's conditions on the shape
      if (l.nstate != 16 || l.width > 4 || l.rank % s.e || l.rank > 8 * s.e || s.k > 128 * s.e ||
          l.dim > 256 * s.e || ssm_decode_xproj_blocks(l.dim, l.nout) < 1)
        return py::none();
    } else if (l.dim != l0.dim || l.nstate != l0.nstate || l.rank != l0.rank ||
               l.width != l0.width || l.eps != l0.eps) {
      return py::none();
    }
    std::memcpy(dst + (size_t)i * sizeof(l.row), l.row, sizeof(l.row));
    ++i;
  }
  return i == count ? py::object(out) : py::object(py::none());
}

py::object block_step(const py::object& block, const py::object& xo, const py::tuple& classes,
                      bool fold, bool rows) {
  Step s;
  Layer l;
  if (!s.open(xo.ptr(), 1, rows ? 64 : 8) || !l.open(s, block.ptr(), Classes(classes)))
    return py::none();
  if (s.batch > 8 && !l.calls_plain) return py::none();
  const at::Tensor& x = *s.x;
  c10::hip::HIPGuard guard(x.get_device());
  void* const st = stream_of(x);
  const float eps = (float)l.eps;
  at::Tensor out = at::empty_like(x);
  const auto bytes = x.options().dtype(at::kByte);
  if (s.batch > 8) {
    const int64_t need = ssm_decode_rows_block_workspace(s.batch, l.dim, l.nout, s.dtype);
    if (need < 1) return py::none();
    at::Tensor ws = at::empty({need}, bytes);
    ok(ssm_decode_rows_block(s.batch, s.k, l.dim, l.nstate, l.rank, l.width, s.dtype, l.row,
                             x.data_ptr(), out.data_ptr(), eps, 1, ws.data_ptr(), need, st));
    return py::cast(out);
  }
  // one workspace: xz, xc, y, the x-projection and (folded) its partial rows
  const int64_t es = 16 / s.e;
  const int64_t nparts = fold ? ssm_decode_xproj_blocks(l.dim, l.nout) : 0;
  auto round = [](int64_t n) { return (n + 255) / 256 * 256; };
  const int64_t row = round(s.batch * l.dim * es), xz_b = round(2 * s.batch * l.dim * es);
  const int64_t par_b = nparts ? round(nparts * s.batch * ((l.nout + 3) / 4 * 4) * 4)
                               : round(s.batch * l.nout * es);
  at::Tensor ws = at::empty({xz_b + 2 * row + par_b}, bytes);
  char* const xz = static_cast<char*>(ws.data_ptr());
  char *const xc = xz + xz_b, *const y = xc + row, *const par = y + row;
  void* const* r = l.row;
  ok(ssm_decode_in_proj_conv(s.batch, l.dim, s.k, l.width, s.dtype, r[SSM_LAYER_IN_PROJ_W],
                             x.data_ptr(), r[SSM_LAYER_NORM_W], eps, r[SSM_LAYER_IN_PROJ_B],
                             r[SSM_LAYER_CONV_W], r[SSM_LAYER_CONV_B], r[SSM_LAYER_CONV_WINDOW], xz,
                             xc, nparts ? r[SSM_LAYER_X_PROJ_W] : nullptr, nparts ? l.nout : 0,
                             nparts ? reinterpret_cast<float*>(par) : nullptr, st));
  if (!nparts)
    ok(ssm_decode_gemv(s.batch, l.nout, l.dim, s.dtype, r[SSM_LAYER_X_PROJ_W], xc, nullptr, 1e-6f,
                       nullptr, nullptr, par, st));
  ok(ssm_decode_ssm_step(s.batch, l.dim, l.nstate, l.rank, s.dtype, par, nparts,
                         r[SSM_LAYER_DT_PROJ_W], r[SSM_LAYER_DT_BIAS], r[SSM_LAYER_LOG_A],
                         r[SSM_LAYER_D], xc, xz, 2 * l.dim,
                         static_cast<float*>(r[SSM_LAYER_STATE]), y, st));
  ok(ssm_decode_gemv(s.batch, s.k, l.dim, s.dtype, r[SSM_LAYER_OUT_PROJ_W], y, nullptr, 1e-6f,
                     r[SSM_LAYER_OUT_PROJ_B], x.data_ptr(), out.data_ptr(), st));
  return py::cast(out);
}

}  // namespace

PYBIND11_MODULE(TORCH_EXTENSION_NAME, m) {
  m.doc() = "Host work of the MI355X decode step (HIP, gfx950)";
  m.def("layer_rows", &layer_rows, py::arg("layers"), py::arg("x"), py::arg("classes"));
  m.def("block_step", &block_step, py::arg("block"), py::arg("x"), py::arg("classes"),
        py::arg("fold"), py::arg("rows"));
}
