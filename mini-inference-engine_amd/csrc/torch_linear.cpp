// The common case of mi355x_fp8_linear from PyTorch, in one native call: the checks, the output
// allocation and the C-ABI call that the Python wrapper otherwise makes one by one.
//
// An eager decode linear takes 6-9 us on the GPU; the wrapper's tensor attribute checks,
// torch.empty, the workspace lookup and a ctypes call with 19 arguments took 13-16 us, so calls
// one after the other were bound by the host.  Anything outside the common case returns None and
// the wrapper goes on as before (it holds the error messages, the copies of strided operands and
// the growing of the workspace), so what is accepted and what is refused is decided there.
//
// The interpreter lock is held over the launches: threads that share a stream share its workspace,
// and their quantizer and GEMM launches must not interleave.
//
// No state lives here but the per-device architecture check (device properties do not change).
// The workspace is the caller's: `buffers` is the wrapper's {(device, stream): byte tensor} dict.
#include <ATen/ATen.h>
#include <ATen/hip/HIPContext.h>
#include <c10/hip/HIPStream.h>
#include <torch/csrc/autograd/python_variable.h>
#include <torch/extension.h>

#include <atomic>
#include <cstring>
#include <stdexcept>
#include <string>

#include "../../include/mi355x_fp8.h"

namespace py = pybind11;

namespace {

bool is_gfx950(int dev) {
  static std::atomic<int> known[64];  // 0 unknown, 1 gfx950, 2 another architecture
  if (dev < 0 || dev >= 64) return false;
  int state = known[dev].load(std::memory_order_relaxed);
  if (state == 0) {
    const char* name = at::cuda::getDeviceProperties(dev)->gcnArchName;
    state = std::strncmp(name, "gfx950", 6) == 0 && (name[6] == '\0' || name[6] == ':') ? 1 : 2;
    known[dev].store(state, std::memory_order_relaxed);
  }
  return state == 1;
}

bool half_type(at::ScalarType t) { return t == at::kBFloat16 || t == at::kHalf; }
int dtype_code(at::ScalarType t) { return t == at::kBFloat16 ? MI355X_FP8_DTYPE_BF16 : MI355X_FP8_DTYPE_F16; }

// The linear's output, or None (nothing launched) for a call the Python wrapper has to handle.
py::object linear(const at::Tensor& x, const at::Tensor& w, const at::Tensor& ws, const py::object& out_dtype,
                  const py::dict& buffers) {
  if (!x.is_cuda() || x.dim() < 2 || w.dim() != 2 || ws.dim() != 2 || !half_type(x.scalar_type()) ||
      w.scalar_type() != at::kFloat8_e4m3fn || ws.scalar_type() != at::kFloat || x.device() != w.device() ||
      x.device() != ws.device())
    return py::none();
  const int64_t k = x.size(-1), n = w.size(0);
  if (k <= 0 || n <= 0 || w.size(1) != k || ws.size(0) != (n + 127) / 128 || ws.size(1) != (k + 127) / 128 ||
      x.numel() == 0 || x.stride(-1) != 1 || w.stride(1) != 1 || (x.dim() > 2 && !x.is_contiguous()))
    return py::none();
  at::ScalarType out_type = x.scalar_type();
  if (!out_dtype.is_none()) {
    if (!THPDtype_Check(out_dtype.ptr())) return py::none();
    out_type = reinterpret_cast<THPDtype*>(out_dtype.ptr())->scalar_type;
    if (!half_type(out_type)) return py::none();
  }
  const int dev = x.device().index();
  if (!is_gfx950(dev)) return py::none();
  const int64_t m = x.numel() / k;
  hipStream_t stream = c10::hip::getCurrentHIPStream(dev).stream();
  // The wrapper's workspace of this device and stream, when it has one of the size.
  const py::tuple key = py::make_tuple(dev, reinterpret_cast<uintptr_t>(stream));
  PyObject* held = PyDict_GetItemWithError(buffers.ptr(), key.ptr());
  if (held == nullptr) {
    if (PyErr_Occurred()) throw py::error_already_set();
    return py::none();
  }
  if (!THPVariable_Check(held)) return py::none();
  const at::Tensor workspace = THPVariable_Unpack(held);
  const size_t bytes = static_cast<size_t>(workspace.numel());
  if (bytes < mi355x_fp8_linear_workspace_bytes(m, n, k, MI355X_FP8_CONFIG_AUTO)) return py::none();
  at::Tensor out = at::empty({m, n}, x.options().dtype(out_type));
  const int status = mi355x_fp8_linear(
      x.data_ptr(), dtype_code(x.scalar_type()), m, k, x.dim() == 2 ? x.stride(0) : k, 1,
      static_cast<const uint8_t*>(w.data_ptr()), w.stride(0), static_cast<const float*>(ws.data_ptr()), ws.stride(0),
      ws.stride(1), n, out.data_ptr(), dtype_code(out_type), n, workspace.data_ptr(), bytes, MI355X_FP8_CONFIG_AUTO,
      stream);
  // A failed launch is reported here: running the call again in the wrapper could succeed and hide
  // it.  Any other status is a refusal, which the wrapper words.
  if (status == MI355X_FP8_ERR_LAUNCH)
    throw std::runtime_error("libmi355x_fp8: " + std::string(mi355x_fp8_status_string(status)) + " (status " +
                             std::to_string(status) + ")");
  if (status != MI355X_FP8_OK) return py::none();
  if (x.dim() > 2) {
    std::vector<int64_t> shape(x.sizes().begin(), x.sizes().end());
    shape.back() = n;
    out = out.view(shape);
  }
  return py::cast(out);
}

}  // namespace

PYBIND11_MODULE(_torch_linear, m) {
  m.def("linear", &linear, "mi355x_fp8_linear for its common case, else None");
}
