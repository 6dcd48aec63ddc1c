// Python module `brainpylib_amd.gpu_ops`: the interface the reference's Python layer expects
// from its `gpu_ops` extension (lib/gpu_ops.cc:179-198): `registrations()` returning
// {target name: PyCapsule("xla._CUSTOM_CALL_TARGET")} and `build_*_descriptor(...)` returning
// the opaque bytes.  It is a thin wrapper over the C ABI of libbrainpylib_amd.so and contains no
// device code.
#include <pybind11/pybind11.h>

#include <string>

#include "../../include/brainpylib_amd.h"

namespace py = pybind11;

namespace {

py::dict Registrations() {
  py::dict dict;
  const int n = bpl_num_targets();
  for (int i = 0; i < n; ++i)
    dict[bpl_target_name(i)] =
        py::capsule(reinterpret_cast<void *>(bpl_target_function(i)), "xla._CUSTOM_CALL_TARGET");
  return dict;
}

// enqueue(target address, stream, opaque, *tensors): the custom call with the tensors' data pointers as its buffers, in
// one call of native code (with ctypes an array of pointers, the call and the query for its error are 2.3 us of host time,
// here 0.6; a step of a small network is bound by them).  Without the interpreter lock, as ctypes calls it.
PyObject *Enqueue(PyObject *, PyObject *const *args, Py_ssize_t n_args) {
  constexpr Py_ssize_t kFixed = 3, kMostBuffers = 16;
  static PyObject *const data_ptr = PyUnicode_InternFromString("data_ptr");
  if (n_args < kFixed || n_args > kFixed + kMostBuffers || !PyBytes_Check(args[2])) {
    PyErr_SetString(PyExc_TypeError, "enqueue(address, stream, opaque, *tensors): up to 16 tensors");
    return nullptr;
  }
  const auto target = reinterpret_cast<bpl_target_fn>(PyLong_AsVoidPtr(args[0]));
  if (target == nullptr) {
    if (!PyErr_Occurred()) PyErr_SetString(PyExc_ValueError, "enqueue: no target");
    return nullptr;
  }
  void *const stream = PyLong_AsVoidPtr(args[1]);
  if (PyErr_Occurred()) return nullptr;
  void *buffers[kMostBuffers] = {};
  for (Py_ssize_t i = kFixed; i < n_args; ++i) {
    PyObject *const address = PyObject_CallMethodNoArgs(args[i], data_ptr);
    if (address == nullptr) return nullptr;
    buffers[i - kFixed] = PyLong_AsVoidPtr(address);
    Py_DECREF(address);
    if (PyErr_Occurred()) return nullptr;
  }
  char *opaque = nullptr;
  Py_ssize_t opaque_len = 0;
  if (PyBytes_AsStringAndSize(args[2], &opaque, &opaque_len) != 0) return nullptr;
  Py_BEGIN_ALLOW_THREADS
  target(stream, buffers, opaque, static_cast<size_t>(opaque_len));
  Py_END_ALLOW_THREADS
  const char *const error = bpl_last_error();  // (per thread, empty unless a target has just failed)
  if (error != nullptr && error[0] != '\0') {
    PyErr_SetString(PyExc_RuntimeError, error);
    bpl_clear_error();
    return nullptr;
  }
  Py_RETURN_NONE;
}
PyMethodDef kEnqueue = {"enqueue", reinterpret_cast<PyCFunction>(reinterpret_cast<void (*)()>(&Enqueue)), METH_FASTCALL,
                        "enqueue(address, stream, opaque, *tensors)"};

// Calls a C-ABI builder with a stack buffer appended to its arguments.
#define BPL_PACK(fn, ...)                                              \
  [&]() {                                                              \
    char bpl_buf_[64];                                                 \
    const size_t bpl_len_ = fn(__VA_ARGS__, bpl_buf_, sizeof(bpl_buf_)); \
    if (bpl_len_ == 0) throw std::runtime_error("descriptor does not fit"); \
    return py::bytes(std::string(bpl_buf_, bpl_len_));                 \
  }()

}  // namespace

PYBIND11_MODULE(gpu_ops, m) {
  m.doc() = "XLA custom-call targets and descriptor builders of brainpylib_amd (gfx950)";
  m.def("registrations", &Registrations);
  m.add_object("enqueue", py::reinterpret_steal<py::object>(PyCFunction_New(&kEnqueue, nullptr)));
  m.def("build_event_csr_batching_descriptor",
        [](uint32_t n_row, uint32_t n_col, uint32_t batch_size, uint32_t values_batch, uint32_t indices_batch,
           uint32_t indptr_batch, uint32_t events_batch, uint32_t nnz, bool transpose) {
          return BPL_PACK(bpl_build_event_csr_batching_descriptor, n_row, n_col, batch_size, values_batch,
                          indices_batch, indptr_batch, events_batch, nnz, transpose ? 1 : 0);
        });
  m.def("build_csr_event_sum_descriptor",
        [](uint32_t pre_size, uint32_t post_size) { return BPL_PACK(bpl_build_csr_event_sum_descriptor, pre_size, post_size); });
  m.def("build_coo_event_sum_descriptor",
        [](uint32_t conn_size, uint32_t post_size) { return BPL_PACK(bpl_build_coo_event_sum_descriptor, conn_size, post_size); });
  m.def("build_coo_atomic_sum_descriptor",
        [](uint32_t conn_size, uint32_t post_size) { return BPL_PACK(bpl_build_coo_atomic_sum_descriptor, conn_size, post_size); });
  m.def("build_coo_atomic_prod_descriptor",
        [](uint32_t conn_size, uint32_t post_size) { return BPL_PACK(bpl_build_coo_atomic_prod_descriptor, conn_size, post_size); });
  m.def("build_csr_event_prod_descriptor",
        [](uint32_t pre_size, uint32_t post_size) { return BPL_PACK(bpl_build_csr_event_prod_descriptor, pre_size, post_size); });
  m.def("build_csr_transpose_descriptor", [](uint32_t n_row, uint32_t n_col, uint32_t nnz) {
    return BPL_PACK(bpl_build_csr_transpose_descriptor, n_row, n_col, nnz);
  });
  m.def("build_twouint_onebool_descriptor", [](uint32_t x, uint32_t y, bool b) {
    return BPL_PACK(bpl_build_twouint_onebool_descriptor, x, y, b ? 1 : 0);
  });
  m.def("build_double_size_descriptor",
        [](uint32_t x, uint32_t y) { return BPL_PACK(bpl_build_double_size_descriptor, x, y); });
  m.def("build_nonzero_descriptor", [](uint32_t event_size, uint32_t batch_size) {
    return BPL_PACK(bpl_build_nonzero_descriptor, event_size, batch_size);
  });
  // prob / weights are taken as double (Python floats): the reference narrows them to float
  m.def("build_jitconn_prob_homo_descriptor", [](uint32_t n_row, uint32_t n_col, uint32_t seed, double prob) {
    return BPL_PACK(bpl_build_jitconn_prob_homo_descriptor, n_row, n_col, seed, prob);
  });
  m.def("build_jitconn_prob_uniform_descriptor",
        [](uint32_t n_row, uint32_t n_col, uint32_t seed, double prob, double w_min, double w_range) {
          return BPL_PACK(bpl_build_jitconn_prob_uniform_descriptor, n_row, n_col, seed, prob, w_min, w_range);
        });
  m.def("build_jitconn_prob_normal_descriptor",
        [](uint32_t n_row, uint32_t n_col, uint32_t seed, double prob, double w_mu, double w_sigma) {
          return BPL_PACK(bpl_build_jitconn_prob_normal_descriptor, n_row, n_col, seed, prob, w_mu, w_sigma);
        });
  m.def("build_matmat_jit_prob_descriptor1",
        [](uint32_t mm, uint32_t k, uint32_t n, uint32_t seed, double log_p, double w1, double w2) {
          return BPL_PACK(bpl_build_matmat_jit_prob_descriptor1, mm, k, n, seed, log_p, w1, w2);
        });
}
