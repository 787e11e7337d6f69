// The oscillator parameters of the D-LinOSS and LinOSS layers from their stored
// form, and the gradients back to it, in one launch each.
//   D-LinOSS (dlinoss.py:249-264): dt = sigmoid(steps), g = relu(G), a clamped to
//     [lo, hi] = (2 + dt g -/+ 2 sqrt(1 + dt g)) / dt^2 as
//     a = lo + relu(A - lo) - relu(A - hi)
//   LinOSS (linoss.py:209-215):    dt = sigmoid(steps), a = relu(A), g = 0
// A few hundred values: the time is launches.  As torch operations the D-LinOSS
// form takes 21 forward launches and about 40 backward, each a host call of about
// 5 us: with them a [8, 1030, 100] layer forward took 134 us and now takes 32 (25 of
// them the layer's own kernel); a [32, 4096, 128] training step took 110 us more.
// The D-LinOSS values are the float operations' own, rounding by rounding (a is
// a difference of nearly equal terms there, and the layer's unfused form, which
// runs them, has to agree with the fused one).  The LinOSS values are formed in
// double and come with what rounding them left, as do both gradients.

#include <hip/hip_runtime.h>

#include <climits>
#include <cstdint>
#include <string>

#include "../../include/ossm_scan.h"
#include "runtime.hpp"

namespace ossm {
namespace {

constexpr int kParamBlock = 128;
constexpr double kClamp = 1e-6;  // the floor of dt^2

// Comparisons are written so that NaN passes through relu and clamp, as in torch.
__device__ __forceinline__ double sigmoid64(double x) { return 1.0 / (1.0 + exp(-x)); }

struct Band {
  float a, g, dt, dt2, dg, root, lo, hi;
};
// project_parameters in its own float operations, none fused
__device__ __forceinline__ Band band_of(float A, float G, float steps) {
#pragma clang fp contract(off)
  Band b;
  b.dt = 1.f / (1.f + expf(-steps));
  b.g = G < 0.f ? 0.f : G;
  const float sq = b.dt * b.dt;
  b.dt2 = sq < 1e-6f ? 1e-6f : sq;
  b.dg = b.dt * b.g;
  const float one = 1.f + b.dg;
  b.root = sqrtf(one < 1e-6f ? 1e-6f : one);
  const float two = 2.f + b.dg, r2 = 2.f * b.root;
  b.lo = (two - r2) / b.dt2;
  b.hi = (two + r2) / b.dt2;
  const float over = A - b.lo, above = A - b.hi;
  b.a = b.lo + (over < 0.f ? 0.f : over) - (above < 0.f ? 0.f : above);
  return b;
}

// out [6][n]: a, g, dt, then (not DAMPED) what rounding each left, from which the
// layer kernels form their coefficients
template <bool DAMPED>
__global__ __launch_bounds__(kParamBlock) void layer_params_fwd_kernel(const float* __restrict__ A,
                                                                       const float* __restrict__ G,
                                                                       const float* __restrict__ steps,
                                                                       float* __restrict__ out, int n) {
  const int p = static_cast<int>(blockIdx.x) * kParamBlock + static_cast<int>(threadIdx.x);
  if (p >= n) return;
  if constexpr (DAMPED) {
    const Band b = band_of(A[p], G[p], steps[p]);
    out[p] = b.a;
    out[n + p] = b.g;
    out[2 * n + p] = b.dt;
  } else {
    const float a = A[p];
    const double dt = sigmoid64(steps[p]);
    const float hi = static_cast<float>(dt);
    out[p] = a < 0.f ? 0.f : a;
    out[n + p] = 0.f;
    out[2 * n + p] = hi;
    out[3 * n + p] = 0.f;
    out[4 * n + p] = 0.f;
    out[5 * n + p] = static_cast<float>(dt - hi);
  }
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
    const Band b = band_of(A[p], G[p], steps[p]);  // which side of the band the forward took
    const bool above_lo = !(A[p] - b.lo <= 0.f), above_hi = !(A[p] - b.hi <= 0.f);
    dt = sigmoid64(steps[p]);
    const double g = b.g, sq = dt * dt, dg = dt * g;
    const double dt2 = sq < kClamp ? kClamp : sq, root = sqrt(1.0 + dg);
    const double lo = (2.0 + dg - 2.0 * root) / dt2, hi = (2.0 + dg + 2.0 * root) / dt2;
    gA = (above_lo ? ga : 0.0) - (above_hi ? ga : 0.0);
    const double glo = above_lo ? 0.0 : ga, ghi = above_hi ? ga : 0.0;
    // 1 + dg >= 1: its clamp never acts
    const double gdg = (glo + ghi) / dt2 + (ghi - glo) * 2.0 / dt2 * 0.5 / root;
    if (!(sq < kClamp)) gdt -= (glo * lo + ghi * hi) / dt2 * 2.0 * dt;
    gdt += gdg * g;
    const double gG = gg + gdg * dt;
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
  if (n < 0 || n > INT_MAX / 8) return set_error(OSSM_ERR_INVALID_ARGUMENT, std::string(what) + ": bad size");
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
