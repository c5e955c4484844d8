// Python bindings of the native host path.
#include <torch/extension.h>

#include "host.h"

namespace py = pybind11;
using namespace aussm_host;

namespace {

// The Python class aussm_amd._lib.AussmError, looked up once (and kept for the life of the process)
PyObject* aussm_error_class() {
  static PyObject* cls = py::object(py::module_::import("aussm_amd._lib").attr("AussmError")).release().ptr();
  return cls;
}

// (y, state) as the caller asked for it
py::object result(const std::pair<Tensor, Tensor>& r, bool want_state) {
  if (want_state) return py::make_tuple(r.first, r.second);
  return py::cast(r.first);
}

}  // namespace

PYBIND11_MODULE(_aussm_host, m) {
  py::register_exception_translator([](std::exception_ptr p) {
    try {
      if (p) std::rethrow_exception(p);
    } catch (const AussmError& e) {
      PyErr_SetString(aussm_error_class(), e.what());
    } catch (const ArgError& e) {
      PyErr_SetString(PyExc_RuntimeError, e.what());
    }
  });
  m.def("unitary_ck", &unitary_ck);
  m.def("unitary_scan", [](const Tensor& u, const Tensor& delta, const Tensor& theta, const Tensor& Bc, const Tensor& Cc, const OptTensor& D,
                           const OptTensor& z, const OptTensor& h0, bool want_state) {
    return result(unitary_scan(u, delta, theta, Bc, Cc, D, z, h0, want_state), want_state);
  });
  m.def("complex_scan", [](const Tensor& u, const Tensor& delta, const Tensor& rho, const Tensor& theta, const Tensor& Bc, const Tensor& Cc,
                           const OptTensor& D, const OptTensor& z, const OptTensor& h0, bool want_state) {
    return result(complex_scan(u, delta, rho, theta, Bc, Cc, D, z, h0, want_state), want_state);
  });
  m.def("selective_scan", [](const Tensor& u, const Tensor& delta, const Tensor& A, const Tensor& B, const Tensor& C, const OptTensor& D,
                             const OptTensor& z, const OptTensor& bias, const OptTensor& h0, bool softplus, bool want_state) {
    return result(selective_scan(u, delta, A, B, C, D, z, bias, softplus, want_state, h0), want_state);
  });
  m.def("operator_supported", &operator_supported);
  m.def("adaptive_operator", &adaptive_operator);
  m.def("aussm_block", [](const Tensor& x, const OptTensor& nw, double eps, bool residual, const Tensor& W_in, const OptTensor& b_in,
                          const Tensor& cw, const OptTensor& cb, const Tensor& W_xp, const Tensor& W_dt, const Tensor& b_dt, const Tensor& xA_w,
                          const Tensor& xA_b, const Tensor& B, const Tensor& C, const Tensor& D, const Tensor& W_out, const OptTensor& b_out,
                          double scale) -> py::object {
    const auto r = aussm_block(x, nw, eps, residual, W_in, b_in, cw, cb, W_xp, W_dt, b_dt, xA_w, xA_b, B, C, D, W_out, b_out, scale);
    if (!r) return py::none();
    return py::make_tuple(r->out, r->u, r->dt, r->xz, r->x_and_bias);
  });
  m.def("mamba_block", &mamba_block);
  m.def("norm_linear", &norm_linear);
}
