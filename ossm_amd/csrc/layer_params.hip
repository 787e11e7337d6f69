// The oscillator parameters of the D-LinOSS and LinOSS layers from their stored
// form, and the gradients back to it, in one launch each.
//   D-LinOSS (dlinoss.py:249-264): dt = sigmoid(steps), g = relu(G), a clamped to
//     [lo, hi] = (2 + dt g -/+ 2 sqrt(1 + dt g)) / dt^2 as
//     a = lo + relu(A - lo) - relu(A - hi)
//   LinOSS (linoss.py:209-215):    dt = sigmoid(steps), a = relu(A), g = 0
// A few hundred values: the time is launches.  As torch operations the D-LinOSS
// form takes 21 forward launches and about 40 backward, each a host call of about
// 5 us: a [8, 1030, 100] layer forward 134 us against 39 here (28 of them the
// layer's own kernel), a [32, 4096, 128] training step 935 against 825.  Each lane works in double and rounds once: lo is a
// difference of nearly equal terms.

#include <hip/hip_runtime.h>

#include <climits>
#include <cstdint>
#include <string>

#include "../../include/ossm_scan.h"
#include "runtime.hpp"

namespace ossm {
namespace {

constexpr int kParamBlock = 128;
constexpr double kClamp = 1e-6;  // the floor of dt^2 and 1 + dt g

// relu and clamp that pass NaN, as torch's do
__device__ __forceinline__ double relu_nan(double x) { return x < 0.0 ? 0.0 : x; }
__device__ __forceinline__ double at_least(double x, double lo) { return x < lo ? lo : x; }
__device__ __forceinline__ double sigmoid64(double x) { return 1.0 / (1.0 + exp(-x)); }

struct Band {
  double dt, g, dt2, dg, root, lo, hi;
};
__device__ __forceinline__ Band band_of(double G, double steps) {
  Band b;
  b.dt = sigmoid64(steps);
  b.g = relu_nan(G);
  b.dt2 = at_least(b.dt * b.dt, kClamp);
  b.dg = b.dt * b.g;
  b.root = sqrt(at_least(1.0 + b.dg, kClamp));
  b.lo = (2.0 + b.dg - 2.0 * b.root) / b.dt2;
  b.hi = (2.0 + b.dg + 2.0 * b.root) / b.dt2;
  return b;
}

// out [3][n]: a, g, dt
template <bool DAMPED>
__global__ __launch_bounds__(kParamBlock) void layer_params_fwd_kernel(const float* __restrict__ A,
                                                                       const float* __restrict__ G,
                                                                       const float* __restrict__ steps,
                                                                       float* __restrict__ out, int n) {
  const int p = static_cast<int>(blockIdx.x) * kParamBlock + static_cast<int>(threadIdx.x);
  if (p >= n) return;
  double a = A[p], g = 0.0, dt;
  if constexpr (DAMPED) {
    const Band b = band_of(G[p], steps[p]);
    a = b.lo + relu_nan(a - b.lo) - relu_nan(a - b.hi);
    g = b.g;
    dt = b.dt;
  } else {
    a = relu_nan(a);
    dt = sigmoid64(steps[p]);
  }
  out[p] = static_cast<float>(a);
  out[n + p] = static_cast<float>(g);
  out[2 * n + p] = static_cast<float>(dt);
}

// grad [3][n]: of A, G (DAMPED), steps; a null upstream gradient is zero
template <bool DAMPED>
__global__ __launch_bounds__(kParamBlock) void layer_params_bwd_kernel(
    const float* __restrict__ A, const float* __restrict__ G, const float* __restrict__ steps,
    const float* __restrict__ ga_in, const float* __restrict__ gg_in, const float* __restrict__ gdt_in,
    float* __restrict__ grad, int n) {
  const int p = static_cast<int>(blockIdx.x) * kParamBlock + static_cast<int>(threadIdx.x);
  if (p >= n) return;
  const double ga = ga_in ? ga_in[p] : 0.0, gg = gg_in ? gg_in[p] : 0.0;
  double gdt = gdt_in ? gdt_in[p] : 0.0;
  const double a = A[p];
  double gA, dt;
  if constexpr (DAMPED) {
    const Band b = band_of(G[p], steps[p]);
    dt = b.dt;
    const bool above_lo = !(a - b.lo <= 0.0), above_hi = !(a - b.hi <= 0.0);
    gA = (above_lo ? ga : 0.0) - (above_hi ? ga : 0.0);
    const double glo = above_lo ? 0.0 : ga, ghi = above_hi ? ga : 0.0;
    const double groot = (ghi - glo) * 2.0 / b.dt2;
    double gdg = (glo + ghi) / b.dt2;
    if (!(1.0 + b.dg < kClamp)) gdg += groot * 0.5 / b.root;
    if (!(b.dt * b.dt < kClamp)) gdt -= (glo * b.lo + ghi * b.hi) / b.dt2 * 2.0 * b.dt;
    gdt += gdg * b.g;
    const double gG = gg + gdg * b.dt;
    grad[n + p] = static_cast<float>(static_cast<double>(G[p]) <= 0.0 ? 0.0 : gG);
  } else {
    dt = sigmoid64(steps[p]);
    gA = a <= 0.0 ? 0.0 : ga;
  }
  grad[p] = static_cast<float>(gA);
  grad[2 * n + p] = static_cast<float>(gdt * dt * (1.0 - dt));
}

int check_params(int damped, const float* A, const float* G, const float* steps, const float* out, int64_t n,
                 const char* what) {
  if (n < 0 || n > INT_MAX / 4) return set_error(OSSM_ERR_INVALID_ARGUMENT, std::string(what) + ": bad size");
  if (n > 0 && (!A || !steps || !out || (damped && !G)))
    return set_error(OSSM_ERR_INVALID_ARGUMENT, std::string(what) + ": null pointer");
  return OSSM_OK;
}

}  // namespace
}  // namespace ossm

using namespace ossm;

extern "C" {

int ossm_layer_params_forward(int damped, const float* A_diag, const float* G_diag, const float* steps,
                              float* out, int64_t ssm, ossm_stream_t stream_v) {
  clear_error();
  if (int rc = check_params(damped, A_diag, G_diag, steps, out, ssm, "layer_params_forward")) return rc;
  if (ssm == 0) return OSSM_OK;
  const int n = static_cast<int>(ssm);
  const dim3 grid(static_cast<unsigned>((n + kParamBlock - 1) / kParamBlock));
  hipStream_t stream = static_cast<hipStream_t>(stream_v);
  if (damped)
    hipLaunchKernelGGL(layer_params_fwd_kernel<true>, grid, dim3(kParamBlock), 0, stream, A_diag, G_diag,
                       steps, out, n);
  else
    hipLaunchKernelGGL(layer_params_fwd_kernel<false>, grid, dim3(kParamBlock), 0, stream, A_diag, G_diag,
                       steps, out, n);
  return launch_check("layer_params_fwd_kernel");
}

int ossm_layer_params_backward(int damped, const float* A_diag, const float* G_diag, const float* steps,
                               const float* grad_a, const float* grad_g, const float* grad_dt, float* grad,
                               int64_t ssm, ossm_stream_t stream_v) {
  clear_error();
  if (int rc = check_params(damped, A_diag, G_diag, steps, grad, ssm, "layer_params_backward")) return rc;
  if (ssm == 0) return OSSM_OK;
  const int n = static_cast<int>(ssm);
  const dim3 grid(static_cast<unsigned>((n + kParamBlock - 1) / kParamBlock));
  hipStream_t stream = static_cast<hipStream_t>(stream_v);
  if (damped)
    hipLaunchKernelGGL(layer_params_bwd_kernel<true>, grid, dim3(kParamBlock), 0, stream, A_diag, G_diag,
                       steps, grad_a, grad_g, grad_dt, grad, n);
  else
    hipLaunchKernelGGL(layer_params_bwd_kernel<false>, grid, dim3(kParamBlock), 0, stream, A_diag, G_diag,
                       steps, grad_a, grad_g, grad_dt, grad, n);
  return launch_check("layer_params_bwd_kernel");
}

}  // extern "C"
