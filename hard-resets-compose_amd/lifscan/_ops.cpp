// C++ autograd functions of the layers over the lifscan C ABI: a layer step costs one Python -> C++
// crossing in the forward and none in the backward.  (A Python autograd function's backward takes
// the interpreter lock on the engine's thread and makes some ten small torch calls.  A step of a
// 1000 x 12800 layer: 122 -> 57 us; 512 x 1024: 116 -> 38 us; a 50000 x 64 parameter fit 254 -> 132
// us.)  They launch the kernels that the Python functions of the same layers launch
// (lifscan/hip_lif.py, hip_affine.py, fit.py); the parameter sums and dL/du0 are finished by one
// kernel (lsh_layer_grads).
// Reference: triton_lif.py:654-687 (LIFTuned), :1003-1026 (LIFAuto), fit.py:15-57 (LIFParamFn),
// :121-153 (LIFSoftScanFn), triton_affine.py:214-246 (LIFAffineFn).
// The entry points' addresses are handed over once from the library the Python package has loaded
// (no link-time dependency, one copy of the library in the process).
#include <torch/extension.h>
#include <c10/core/DeviceGuard.h>
#include <c10/hip/HIPStream.h>

#include <algorithm>
#include <array>
#include <cstdint>
#include <map>
#include <mutex>
#include <string>
#include <vector>

#include "lifscan_hip.h"

namespace {

using torch::Tensor;
using torch::autograd::AutogradContext;
using torch::autograd::variable_list;

// The library's entry points, by the declarations of the C ABI header.
struct Entry {
#define LSH_ENTRIES(X)                                                                            \
  X(lsh_status_string)                                                                            \
  X(lsh_lif_layer_fwd)                                                                            \
  X(lsh_lif_layer_bwd)                                                                            \
  X(lsh_lif_layer_bwd_workspace)                                                                  \
  X(lsh_lif_layer_partials)                                                                       \
  X(lsh_lif_scan_warm_any_fwd)                                                                    \
  X(lsh_lif_scan_warm_any_workspace)                                                              \
  X(lsh_lif_scan_lookback_any_bwd)                                                                \
  X(lsh_lif_scan_lookback_any_bwd_workspace)                                                      \
  X(lsh_lif_param_bwd)                                                                            \
  X(lsh_lif_param_partials)                                                                       \
  X(lsh_layer_grads)                                                                              \
  X(lsh_aff_serial_fwd)                                                                           \
  X(lsh_aff_scan_fwd)                                                                             \
  X(lsh_aff_bwd)                                                                                  \
  X(lsh_soft_bwd)                                                                                 \
  X(lsh_soft_bwd_workspace)                                                                       \
  X(lsh_soft_bwd_partials)
#define LSH_MEMBER(name) decltype(&::name) name = nullptr;
  LSH_ENTRIES(LSH_MEMBER)
#undef LSH_MEMBER
} g;
bool g_set = false;

void set_entry_points(const std::map<std::string, int64_t>& addresses) {
#define LSH_SET(name) g.name = reinterpret_cast<decltype(&::name)>(addresses.at(#name));
  LSH_ENTRIES(LSH_SET)
#undef LSH_SET
  g_set = true;
}

void check(int rc, const char* what) {
  if (rc == 0) return;
  const std::string msg = std::string(what) + ": " + g.lsh_status_string(rc) + " (status " +
                          std::to_string(rc) + ")";
  // argument errors are ValueError on the Python side, as the ctypes path raises them
  if (rc == -1 || rc == -2 || rc == -3) TORCH_CHECK_VALUE(false, msg);
  TORCH_CHECK(false, msg);
}

void* stream_of(const Tensor& t) {
  return static_cast<void*>(c10::hip::getCurrentHIPStream(t.device().index()).stream());
}
float* fp(const Tensor& t) { return t.defined() ? t.data_ptr<float>() : nullptr; }
double* dp(const Tensor& t) { return t.defined() ? t.data_ptr<double>() : nullptr; }
Tensor workspace(size_t bytes, const Tensor& like) {
  if (bytes == 0) return Tensor();
  return torch::empty({(int64_t)std::max<size_t>(bytes, 256)}, like.options().dtype(torch::kUInt8));
}
void* raw(const Tensor& t) { return t.defined() ? t.data_ptr() : nullptr; }
Tensor partials(int64_t rows, int64_t cols, const Tensor& like) {
  return torch::empty({std::max<int64_t>(rows, 1), cols}, like.options().dtype(torch::kFloat64));
}
using Param = c10::optional<Tensor>;  // a parameter that wants a gradient, or none
bool wants(const Param& t) { return t.has_value() && t->requires_grad(); }

void check_layer(const Tensor& I, const Tensor& u0) {
  TORCH_CHECK(g_set, "lifscan ops: entry points not set");
  TORCH_CHECK_VALUE(I.dim() == 2 && I.is_cuda() && I.scalar_type() == torch::kFloat32,
                    "I must be a float32 [T, N] GPU tensor");
  TORCH_CHECK_VALUE(u0.dim() == 1 && u0.size(0) == I.size(1) && u0.is_contiguous() &&
                        u0.scalar_type() == torch::kFloat32 && u0.device() == I.device(),
                    "u0 must be a float32 [N] tensor on I's device");
}

// A saved tensor as the kernels read it.  A saved-tensor hook may hand back another one than it was
// given (off the GPU, in half precision, with other strides), so what the forward's checks showed is
// checked again before its address is used.
Tensor unpacked(const Tensor& t, torch::IntArrayRef sizes, const Tensor& like) {
  TORCH_CHECK_VALUE(t.defined() && t.is_cuda() && t.device() == like.device() &&
                        t.scalar_type() == torch::kFloat32 && t.sizes() == sizes,
                    "a saved tensor was unpacked to something else than the float32 ", sizes,
                    " tensor on ", like.device(), " that was saved");
  return t.contiguous();
}

// The workspace of the most recent look-back adjoint run here, whose header counts the bounded waits
// that gave up (hip_lif.last_lookback_timeouts), and how many have run, by which the Python side
// tells which of the two ran last.  Set from the engine's threads; left to the process at its end,
// when the device may be gone.
struct Lookback {
  std::mutex lock;
  Param ws;
  int64_t runs = 0;
};
Lookback& lookback() {
  static Lookback* l = new Lookback;
  return *l;
}
void note_lookback(const Tensor& ws) {
  Param old = ws;  // freed outside the lock
  const std::lock_guard<std::mutex> guard(lookback().lock);
  std::swap(lookback().ws, old);
  ++lookback().runs;
}
Param last_lookback() {
  const std::lock_guard<std::mutex> guard(lookback().lock);
  return lookback().ws;
}
int64_t lookback_runs() {
  const std::lock_guard<std::mutex> guard(lookback().lock);
  return lookback().runs;
}

// The scaled column sums of the partials (undefined: none) and dL/du0 = beta * Lam[0], in one launch.
struct Small {
  Tensor sums, du0;
};
Small finish(const Tensor& parts, double s0, double s1, double s2, const Tensor& Lam, double beta,
             bool want_du0) {
  Small out;
  if (parts.defined()) out.sums = torch::empty({parts.size(1)}, Lam.options());
  if (want_du0) out.du0 = torch::empty({Lam.size(1)}, Lam.options());
  if (!parts.defined() && !want_du0) return out;
  check(g.lsh_layer_grads(parts.defined() ? parts.data_ptr<double>() : nullptr,
                          parts.defined() ? parts.size(0) : 0, parts.defined() ? (int)parts.size(1) : 1,
                          s0, s1, s2, fp(out.sums), fp(Lam), Lam.size(1), (float)beta, fp(out.du0),
                          stream_of(Lam)),
        "lsh_layer_grads");
  return out;
}

// A backward's result: the gradients of I, u0 and the (up to) three parameter tensors that want one,
// then undefined for the forward's other arguments.
variable_list grads_of(const Small& s, const Tensor& Lam, const std::array<int64_t, 3>& want,
                       size_t arguments) {
  variable_list out(arguments);
  out[0] = Lam;
  out[1] = s.du0;
  for (int k = 0; k < 3; ++k)
    if (want[k]) out[2 + k] = s.sums[k];
  return out;
}

// ---------------------------------------------------------------------------------------------
// Hard-reset LIF: S, with gradients for I, u0 and (where given as tensors) beta, theta, u_r.
// warm_C > 0: warm-started chunks of that length (few neurons, long T), which keep U and S for the
// look-back adjoint; else the layer pair.
struct LIFLayer : public torch::autograd::Function<LIFLayer> {
  static Tensor forward(AutogradContext* ctx, const Tensor& I_in, const Tensor& u0, const Param& bt,
                        const Param& tt, const Param& rt, double beta, double theta, double u_r,
                        double alpha, const Tensor& hdr, int64_t warm_C, int64_t warm_W) {
    const Tensor I = I_in.contiguous();
    const c10::DeviceGuard guard(I.device());
    const int64_t T = I.size(0), N = I.size(1);
    auto S = torch::empty_like(I);
    if (warm_C > 0) {
      auto U = torch::empty_like(I);
      const size_t nb = g.lsh_lif_scan_warm_any_workspace(T, N, (int)warm_C);
      const Tensor ws = workspace(nb, I);
      check(g.lsh_lif_scan_warm_any_fwd(fp(I), fp(u0), fp(U), fp(S), T, N, (float)beta, (float)theta,
                                        (float)u_r, (int)warm_C, (int)warm_W, raw(ws), nb, stream_of(I)),
            "lsh_lif_scan_warm_any_fwd");
      ctx->save_for_backward({I, u0, U, S});
    } else {
      auto ST = torch::empty({(T + 31) / 32, N}, I.options());
      check(g.lsh_lif_layer_fwd(fp(I), fp(u0), fp(ST), fp(S), T, N, (float)beta, (float)theta,
                                (float)u_r, raw(hdr), (size_t)hdr.numel(), stream_of(I)),
            "lsh_lif_layer_fwd");
      ctx->save_for_backward({I, ST});
    }
    ctx->saved_data["c"] = std::vector<double>{beta, theta, u_r, alpha};
    ctx->saved_data["n"] = std::vector<int64_t>{wants(u0), wants(bt), wants(tt), wants(rt)};
    return S;
  }

  static variable_list backward(AutogradContext* ctx, variable_list grads) {
    const auto saved = ctx->get_saved_variables();
    const auto c = ctx->saved_data["c"].toDoubleVector();
    const auto n = ctx->saved_data["n"].toIntVector();
    const c10::DeviceGuard guard(grads[0].device());
    const Tensor gS = grads[0].contiguous();  // of the spikes' shape and device (the engine's check)
    const int64_t T = gS.size(0), N = gS.size(1);
    const Tensor I = unpacked(saved[0], gS.sizes(), gS);
    const float beta = (float)c[0], theta = (float)c[1], u_r = (float)c[2], alpha = (float)c[3];
    auto Lam = torch::empty_like(I);
    const bool sums = n[1] || n[2] || n[3];
    Tensor parts;
    if (saved.size() == 4) {
      const Tensor u0 = unpacked(saved[1], {N}, gS), U = unpacked(saved[2], gS.sizes(), gS),
                   S = unpacked(saved[3], gS.sizes(), gS);
      const size_t nb = g.lsh_lif_scan_lookback_any_bwd_workspace(T, N);
      const Tensor ws = workspace(nb, I);
      if (sums) {
        parts = partials(g.lsh_lif_param_partials(T, N, 4, 16), 3, I);
        check(g.lsh_lif_param_bwd(fp(I), fp(u0), fp(U), fp(S), fp(gS), fp(Lam), dp(parts), T, N, beta,
                                  theta, u_r, alpha, 4, 16, raw(ws), nb, stream_of(I)),
              "lsh_lif_param_bwd");
      } else {
        check(g.lsh_lif_scan_lookback_any_bwd(fp(I), fp(u0), fp(U), fp(S), fp(gS), nullptr, fp(Lam), T,
                                              N, beta, theta, u_r, alpha, 1, 16, raw(ws), nb,
                                              stream_of(I)),
              "lsh_lif_scan_lookback_any_bwd");
      }
      note_lookback(ws);
    } else {
      const Tensor ST = unpacked(saved[1], {(T + 31) / 32, N}, gS);
      const size_t nb = g.lsh_lif_layer_bwd_workspace(T, N);
      const Tensor ws = workspace(nb, I);
      if (sums) parts = partials(g.lsh_lif_layer_partials(T, N), 3, I);
      check(g.lsh_lif_layer_bwd(fp(I), fp(ST), fp(gS), fp(Lam), dp(parts), T, N, beta, theta, u_r,
                                alpha, raw(ws), nb, stream_of(I)),
            "lsh_lif_layer_bwd");
      if (nb) note_lookback(ws);
    }
    const Small s = finish(parts, 1.0, -1.0, beta, Lam, beta, n[0] != 0);
    return grads_of(s, Lam, {n[1], n[2], n[3]}, 12);
  }
};

Tensor lif_layer(const Tensor& I, const Tensor& u0, const Param& bt,
                 const Param& tt, const Param& rt, double beta,
                 double theta, double u_r, double alpha, const Tensor& hdr, int64_t C, int64_t W) {
  check_layer(I, u0);
  return LIFLayer::apply(I, u0, bt, tt, rt, beta, theta, u_r, alpha, hdr, C, W);
}

// Spikes alone, outside autograd.
Tensor lif_spikes(const Tensor& I_in, const Tensor& u0, double beta, double theta, double u_r,
                  const Tensor& hdr) {
  check_layer(I_in, u0);
  const Tensor I = I_in.detach().contiguous();
  const c10::DeviceGuard guard(I.device());
  auto S = torch::empty_like(I);
  check(g.lsh_lif_layer_fwd(fp(I), fp(u0), nullptr, fp(S), I.size(0), I.size(1), (float)beta,
                            (float)theta, (float)u_r, raw(hdr), (size_t)hdr.numel(), stream_of(I)),
        "lsh_lif_layer_fwd");
  return S;
}

// ---------------------------------------------------------------------------------------------
// Affine reset (soft = false) and soft reset: the two-level scan (C > 0) or the serial sweep (C = 0),
// and the adjoint with the gradients for I, u0, beta[, gamma, delta].  code, Cb: lsh_aff_bwd's mode and
// chunk, or the soft adjoint's chunk in Cb.
struct AffLayer : public torch::autograd::Function<AffLayer> {
  static Tensor forward(AutogradContext* ctx, const Tensor& I_in, const Tensor& u0, const Param& bt,
                        const Param& gt, const Param& dt, std::vector<double> c, bool soft,
                        const Tensor& ws, int64_t C, int64_t K, int64_t code, int64_t Cb) {
    const Tensor I = I_in.contiguous();
    const c10::DeviceGuard guard(I.device());
    const int64_t T = I.size(0), N = I.size(1);
    const double beta = c[0], theta = c[1], gamma = c[2], delta = c[3];
    auto U = torch::empty_like(I), S = torch::empty_like(I);
    if (C > 0) {
      check(g.lsh_aff_scan_fwd(fp(I), fp(u0), fp(U), fp(S), T, N, (float)beta, (float)theta,
                               (float)gamma, (float)delta, (float)(gamma * theta + delta), (int)C, (int)K,
                               0, raw(ws), (size_t)ws.numel(), stream_of(I)),
            "lsh_aff_scan_fwd");
    } else {
      check(g.lsh_aff_serial_fwd(fp(I), fp(u0), fp(U), fp(S), T, N, (float)beta, (float)theta,
                                 (float)gamma, (float)delta, stream_of(I)),
            "lsh_aff_serial_fwd");
    }
    if (soft)
      ctx->save_for_backward({I, u0, U});
    else
      ctx->save_for_backward({I, u0, U, S});
    ctx->saved_data["c"] = c;
    ctx->saved_data["n"] = std::vector<int64_t>{wants(u0), wants(bt), wants(gt), wants(dt), code, Cb};
    return S;
  }

  static variable_list backward(AutogradContext* ctx, variable_list grads) {
    const auto saved = ctx->get_saved_variables();
    const auto c = ctx->saved_data["c"].toDoubleVector();
    const auto n = ctx->saved_data["n"].toIntVector();
    const c10::DeviceGuard guard(grads[0].device());
    const Tensor gS = grads[0].contiguous();  // of the spikes' shape and device (the engine's check)
    const int64_t T = gS.size(0), N = gS.size(1);
    const Tensor I = unpacked(saved[0], gS.sizes(), gS), u0 = unpacked(saved[1], {N}, gS),
                 U = unpacked(saved[2], gS.sizes(), gS);
    const double beta = c[0], theta = c[1], gamma = c[2], alpha = c[4];
    const int code = (int)n[4], Cb = (int)n[5];
    auto Lam = torch::empty_like(I);
    Tensor parts;
    if (saved.size() == 3) {  // soft reset
      const size_t nb = g.lsh_soft_bwd_workspace(T, N, Cb);
      const Tensor ws = workspace(nb, I);
      if (n[1]) parts = partials(g.lsh_soft_bwd_partials(T, N, Cb), 1, I);
      check(g.lsh_soft_bwd(fp(I), fp(u0), fp(U), nullptr, fp(gS), fp(Lam), dp(parts), T, N, beta,
                           (float)theta, (float)alpha, Cb, raw(ws), nb, stream_of(I)),
            "lsh_soft_bwd");
      const Small s = finish(parts, 1.0, 0.0, 0.0, Lam, beta, n[0] != 0);
      return grads_of(s, Lam, {n[1], 0, 0}, 12);
    }
    const Tensor S = unpacked(saved[3], gS.sizes(), gS);
    const size_t nb = code >= 3 ? g.lsh_lif_scan_lookback_any_bwd_workspace(T, N) : 0;
    const Tensor ws = workspace(nb, I);
    parts = partials(g.lsh_lif_param_partials(T, N, code, Cb), 3, I);
    check(g.lsh_aff_bwd(fp(I), fp(u0), fp(U), fp(S), fp(gS), fp(Lam), dp(parts), T, N, (float)beta,
                        (float)theta, (float)gamma, (float)alpha, code, Cb, raw(ws), nb, stream_of(I)),
          "lsh_aff_bwd");
    if (nb) note_lookback(ws);
    const bool sums = n[1] || n[2] || n[3];
    const Small s = finish(sums ? parts : Tensor(), 1.0, beta, beta, Lam, beta, n[0] != 0);
    return grads_of(s, Lam, {n[1], n[2], n[3]}, 12);
  }
};

Tensor aff_layer(const Tensor& I, const Tensor& u0, const Param& bt,
                 const Param& gt, const Param& dt,
                 std::vector<double> c, bool soft, const Tensor& ws, int64_t C, int64_t K, int64_t code,
                 int64_t Cb) {
  check_layer(I, u0);
  return AffLayer::apply(I, u0, bt, gt, dt, c, soft, ws, C, K, code, Cb);
}

// The values of one-element floating-point tensors of one device and type, in one copy.
std::vector<double> read_scalars(const std::vector<Tensor>& ts) {
  const torch::NoGradGuard no_grad;
  std::vector<Tensor> flat;
  for (const auto& t : ts) flat.push_back(t.reshape({1}));
  const Tensor host = torch::cat(flat).to(torch::kCPU).to(torch::kFloat64);
  const double* p = host.data_ptr<double>();
  return std::vector<double>(p, p + host.numel());
}

}  // namespace

PYBIND11_MODULE(TORCH_EXTENSION_NAME, m) {
  m.doc() = "C++ autograd functions of the lifscan layers over the lifscan C ABI";
  m.def("set_entry_points", &set_entry_points, "addresses of the C-ABI entry points, by name");
  m.def("lif_layer", &lif_layer, "hard-reset LIF layer: S");
  m.def("lif_spikes", &lif_spikes, "hard-reset LIF spikes outside autograd");
  m.def("aff_layer", &aff_layer, "affine- or soft-reset LIF layer: S");
  m.def("last_lookback", &last_lookback, "workspace of the most recent look-back adjoint here, or None");
  m.def("lookback_runs", &lookback_runs, "look-back adjoints run here so far");
  m.def("read_scalars", &read_scalars, "values of one-element tensors in one copy");
}
