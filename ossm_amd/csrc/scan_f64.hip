// The complex128 scans on gfx950 that the reference's device kernels dispatch
// besides complex64: D-LinOSS (dlinoss_imex1_cuda.cu:196, 234, and the imex2 /
// im / ex siblings), selective D-LinOSS (sdlinoss_imex1_cuda.cu:232, 271, and
// siblings) and the LinOSS scan (linoss_scan_cuda.cu:139).
//
// Time is cut into chunks so that the whole device works on a sequence (a lane
// that walks all of it leaves most CUs idle and pays a memory round trip every
// few steps).  Two launches, no wait between workgroups, every sum in a fixed
// order, so the results repeat bit for bit:
//   1. chunk64_{fwd,bwd}_kernel: each (chunk, channel) scans its steps from a
//      zero carry and stores where it ends (and, for parameters that vary over
//      time, the product of its transitions);
//   2. scan64_{fwd,bwd}_kernel: each (chunk, channel) folds the aggregates of
//      the chunks before it (after it, in reverse) into its carry, with the
//      chunk transition M^CL formed once per lane by binary powering (or the
//      stored products; a carry that is not finite is walked step by step
//      instead), and walks its steps again from that carry, writing the
//      outputs.  Consecutive lanes own consecutive channels, so every load and
//      store of a wave is one contiguous run.
// Bound by HBM: a forward reads bu twice (the second time largely from the
// last-level cache) and writes the states, 64 B per state-step of complex128
// D-LinOSS against the 48 it cannot do without; the backward 96 against 80.
// Chunk count and measured figures: chunks64.
// With one chunk (short sequences, channels enough to fill the device, or under
// stream capture when the workspace would have to grow) step 2 alone is the plain
// sequential scan.
//
// Selective D-LinOSS: recurrence and chain rule of the complex64 kernels
// (sdlinoss_<v>.cpp forward kernels, backward kernels sdlinoss_imex1.cpp:186-220,
// sdlinoss_imex2.cpp:178-221, sdlinoss_im.cpp:176-225,
// sdlinoss_ex.cpp:163-189), in double, with the division by S kept as a
// division:
//   dt = clamp(step, 1e-6, 1), comb = -a x + bu, tmpw = alpha w + dt^2 comb,
//   w' = tmpw / S, x' = x + w'.
// Parameter gradients broadcast over time are summed over a chunk's steps in
// the lane and over the chunks (and batch rows) afterwards, in row order.
//
// LinOSS: s_t = M s_{t-1} + b_t with a complex 2x2 M per oscillator
// (linoss_scan.cpp:11-96); backward g_t = grad_t + M^H g_{t+1}, grad_b_t = g_t,
// grad_M_ij = sum over (b, t) of g_i,t conj(s_j,t-1) (linoss.py:83-151), summed
// over a chunk's steps in the lane and over chunks and batch rows afterwards.

#include <hip/hip_runtime.h>

#include <algorithm>
#include <climits>
#include <cmath>
#include <cstdint>
#include <string>

#include "../../include/ossm_scan.h"
#include "runtime.hpp"
#include "scan_device.hpp"

namespace ossm {
namespace {

constexpr double kDtMin64 = 1e-6;
constexpr double kDtMax64 = 1.0;
constexpr double kClampMin64 = 1e-6;
constexpr int kBlock64 = 256;

// One parameter [La, Ba, M]: element (t, channel ch = b M + m) at
// p[t * t_stride + (by_channel ? ch : m)].
struct View64 {
  const double* p;
  long long t_stride;
  int by_channel;
};

struct Params64 {
  View64 v[3];  // a, g, step
  int M;
};

__device__ __forceinline__ double at64(const View64& v, int t, int ch, int m) {
  return v.p[static_cast<size_t>(t) * v.t_stride + (v.by_channel ? ch : m)];
}

template <int V>
__device__ __forceinline__ double alpha64(double dt, double g) {
  if constexpr (V == OSSM_DLINOSS_IMEX2 || V == OSSM_DLINOSS_EX) return 1.0 - dt * g;
  else return 1.0;
}

template <int V>
__device__ __forceinline__ double s_raw64(double dt, double g, double a) {
  if constexpr (V == OSSM_DLINOSS_IMEX1) return 1.0 + dt * g;
  else if constexpr (V == OSSM_DLINOSS_IMEX2) return 1.0 + dt * dt * a;
  else if constexpr (V == OSSM_DLINOSS_IM) return 1.0 + dt * g + dt * dt * a;
  else return 1.0;
}

__device__ __forceinline__ double dt64(double step_raw) {
  return fmin(fmax(step_raw, kDtMin64), kDtMax64);
}

// A state or adjoint: a complex 2-vector (s0.re, s0.im, s1.re, s1.im).
struct St {
  double x, y, z, w;
};
__device__ __forceinline__ St st_zero() { return {0.0, 0.0, 0.0, 0.0}; }
__device__ __forceinline__ St st_add(St a, St b) {
  return {a.x + b.x, a.y + b.y, a.z + b.z, a.w + b.w};
}
__device__ __forceinline__ St st_apply(const RMatD& m, St s) {
  return {m.a * s.x + m.b * s.z, m.a * s.y + m.b * s.w, m.c * s.x + m.d * s.z,
          m.c * s.y + m.d * s.w};
}
__device__ __forceinline__ St st_apply(const CMatD& m, St s) {
  return {m.ar * s.x - m.ai * s.y + m.br * s.z - m.bi * s.w,
          m.ar * s.y + m.ai * s.x + m.br * s.w + m.bi * s.z,
          m.cr * s.x - m.ci * s.y + m.dr * s.z - m.di * s.w,
          m.cr * s.y + m.ci * s.x + m.dr * s.w + m.di * s.z};
}
__device__ __forceinline__ RMatD adjoint64(const RMatD& m) { return {m.a, m.c, m.b, m.d}; }
__device__ __forceinline__ CMatD adjoint64(const CMatD& m) {
  return {m.ar, -m.ai, m.cr, -m.ci, m.br, -m.bi, m.dr, -m.di};
}
// m^n, n >= 1
template <class Mat>
__device__ __forceinline__ Mat pow64(Mat b, int n) {
  Mat r = mat_identity(b);
  while (n > 0) {
    if (n & 1) r = mat_mul(r, b);
    n >>= 1;
    if (n) b = mat_mul(b, b);
  }
  return r;
}
__device__ __forceinline__ St load_st(const double2* p) {
  const double2 a = p[0], b = p[1];
  return {a.x, a.y, b.x, b.y};
}
__device__ __forceinline__ void store_st(double2* p, St s) {
  p[0] = make_double2(s.x, s.y);
  p[1] = make_double2(s.z, s.w);
}

// ---- models: one step of each recurrence, its adjoint and its gradients -----
// kVarying: the parameters may change every step (no matrix power; the local
// pass stores the product of the chunk's transitions).  Time sums: kSums
// doubles per (chunk, channel), part[(chunk nc + ch) kSums + i].

// Where a scan is cut into chunks (Model::kFwd, kBwd): from `min_len` steps on, and
// where 2048 waves give each sequence at least `min_chunks`, or `min_chunks_big` once
// the call moves `big` bytes.  Below, the second launch, the fold and the second
// read of the inputs cost more than the idle units; the bytes matter because the
// second read comes from the last-level cache (256 MB) up to there, as do all of a
// repeated call's.
struct Chunking {
  int64_t min_len, min_chunks, big, min_chunks_big;
};
constexpr int64_t kMb = 1 << 20;

// Selective D-LinOSS.
// Where parameter p's gradient goes (mode[p]): 0 = per element at
// out[t * nc + ch] (full shape); 1 = summed over time; 2 = per element, to be
// summed over the batch rows afterwards.
struct Grads64 {
  double* out[3];
  int mode[3];
};

template <int V>
struct Sdl64 {
  static constexpr bool kVarying = true;
  static constexpr int kSums = 3;
  static constexpr Chunking kFwd{64, 10, 256 * kMb, 5}, kBwd{40, 4, 0, 4}, kBwdConstant{40, 3, 0, 3};
  using Params = Params64;
  using Mat = RMatD;
  using Grads = Grads64;
  using In = double2;
  struct Coef {
    double a, g, step_raw, dt, dt2, alpha, s_raw, S;
  };
  static __device__ __forceinline__ int width(const Params& prm) { return prm.M; }
  static __device__ __forceinline__ Coef coef(const Params& prm, int t, int ch, int m) {
    Coef k;
    k.a = at64(prm.v[0], t, ch, m);
    k.g = at64(prm.v[1], t, ch, m);
    k.step_raw = at64(prm.v[2], t, ch, m);
    k.dt = dt64(k.step_raw);
    k.dt2 = k.dt * k.dt;
    k.alpha = alpha64<V>(k.dt, k.g);
    k.s_raw = s_raw64<V>(k.dt, k.g, k.a);
    k.S = fmax(k.s_raw, kClampMin64);
    return k;
  }
  static __device__ __forceinline__ In load_in(const double2* in, size_t e) { return in[e]; }
  static __device__ __forceinline__ St step(const Coef& k, St s, In b) {
    double tr = k.alpha * s.x + k.dt2 * (-k.a * s.z + b.x);
    double ti = k.alpha * s.y + k.dt2 * (-k.a * s.w + b.y);
    if constexpr (V != OSSM_DLINOSS_EX) {
      tr /= k.S;
      ti /= k.S;
    }
    return {tr, ti, s.z + tr, s.w + ti};
  }
  static __device__ __forceinline__ Mat matrix(const Coef& k) {
    double c0 = k.alpha, c1 = -k.dt2 * k.a;
    if constexpr (V != OSSM_DLINOSS_EX) {
      c0 /= k.S;
      c1 /= k.S;
    }
    return {c0, c1, c0, 1.0 + c1};
  }
  // the upstream gradient enters through x
  static __device__ __forceinline__ St mu(St y, In go) { return {y.x, y.y, y.z + go.x, y.w + go.y}; }
  // carry to the previous state: d/dw_prev = alpha gt, d/dx_prev = lx - dt^2 a gt
  static __device__ __forceinline__ St rev(const Coef& k, St m) {
    double gr = m.x + m.z, gi = m.y + m.w;
    if constexpr (V != OSSM_DLINOSS_EX) {
      gr /= k.S;
      gi /= k.S;
    }
    return {k.alpha * gr, k.alpha * gi, m.z - k.dt2 * k.a * gr, m.w - k.dt2 * k.a * gi};
  }
  // one step's gradients, bu's streamed (written once, read by a later launch:
  // 3 to 6 % of the backward; the states' two half-lines per lane lose by it):
  // bu, then a, g, step (tmpw = alpha w + dt^2 (-a x + bu))
  static __device__ __forceinline__ void grads(const Coef& k, St m, St sp, In b, double2* gin, size_t e,
                                               double* acc, const Grads& dst) {
    const double gwr = m.x + m.z, gwi = m.y + m.w;  // w.r.t. the new w, through both components
    const double combr = -k.a * sp.z + b.x, combi = -k.a * sp.w + b.y;
    double gdt = 0.0, gA = 0.0, gG = 0.0;
    double gtr = gwr, gti = gwi;  // w.r.t. tmpw
    if constexpr (V != OSSM_DLINOSS_EX) {
      const double tmpr = k.alpha * sp.x + k.dt2 * combr, tmpi = k.alpha * sp.y + k.dt2 * combi;
      gtr = gwr / k.S;
      gti = gwi / k.S;
      const double gS = k.s_raw > kClampMin64 ? -(gwr * tmpr + gwi * tmpi) / (k.S * k.S) : 0.0;
      if constexpr (V == OSSM_DLINOSS_IMEX1) {
        gdt = gS * k.g;
        gG = gS * k.dt;
      } else if constexpr (V == OSSM_DLINOSS_IMEX2) {
        gdt = gS * (2.0 * k.dt * k.a);
        gA = gS * k.dt2;
      } else {
        gdt = gS * (k.g + 2.0 * k.dt * k.a);
        gA = gS * k.dt2;
        gG = gS * k.dt;
      }
    }
    if constexpr (V == OSSM_DLINOSS_IMEX2 || V == OSSM_DLINOSS_EX) {
      gdt += gtr * (-k.g * sp.x + 2.0 * k.dt * combr) + gti * (-k.g * sp.y + 2.0 * k.dt * combi);
      gG += gtr * (-k.dt * sp.x) + gti * (-k.dt * sp.y);
    } else {
      gdt += gtr * (2.0 * k.dt * combr) + gti * (2.0 * k.dt * combi);
    }
    gA += gtr * (-k.dt2 * sp.z) + gti * (-k.dt2 * sp.w);
    stream_store(gin + e, make_double2(gtr * k.dt2, gti * k.dt2));
    const double gp[3] = {gA, gG, (k.step_raw > kDtMin64 && k.step_raw < kDtMax64) ? gdt : 0.0};
#pragma unroll
    for (int p = 0; p < 3; ++p) {
      if (dst.mode[p] == 1) acc[p] += gp[p];
      else dst.out[p][e] = gp[p];
    }
  }
  // the time sums of parameter p go where its reduction reads them
  static __device__ __forceinline__ void store_sums(const Grads& dst, double*, size_t row, const double* acc) {
#pragma unroll
    for (int p = 0; p < 3; ++p)
      if (dst.mode[p] == 1) dst.out[p][row] = acc[p];
  }
};

// LinOSS: states [L, nc, 2] and b [L, nc, 2], channel ch = b P + p.
struct Lin64Params {
  const double2* m[4];  // m11, m12, m21, m22, [P] each
  int P;
};
struct NoGrads64 {};

struct Lin64 {
  static constexpr bool kVarying = false;
  static constexpr int kSums = 8;  // grad_m's (re, im) of m11, m12, m21, m22
  static constexpr Chunking kFwd{100, 10, 256 * kMb, 5}, kBwd{100, 12, 300 * kMb, 8};
  using Params = Lin64Params;
  using Mat = CMatD;
  using Grads = NoGrads64;
  using In = St;
  using Coef = CMatD;
  static __device__ __forceinline__ int width(const Params& prm) { return prm.P; }
  static __device__ __forceinline__ Coef coef(const Params& prm, int, int, int p) {
    const double2 a = prm.m[0][p], b = prm.m[1][p], c = prm.m[2][p], d = prm.m[3][p];
    return {a.x, a.y, b.x, b.y, c.x, c.y, d.x, d.y};
  }
  static __device__ __forceinline__ In load_in(const double2* in, size_t e) { return load_st(in + 2 * e); }
  static __device__ __forceinline__ St step(const Coef& k, St s, In b) { return st_add(st_apply(k, s), b); }
  static __device__ __forceinline__ Mat matrix(const Coef& k) { return k; }
  static __device__ __forceinline__ St mu(St y, In go) { return st_add(go, y); }
  static __device__ __forceinline__ St rev(const Coef& k, St g) { return st_apply(adjoint64(k), g); }
  // grad_b_t = g_t; grad_m_ij += g_i conj(s_j,t-1)
  static __device__ __forceinline__ void grads(const Coef&, St g, St sp, In, double2* gin, size_t e,
                                               double* acc, const Grads&) {
    store_st(gin + 2 * e, g);
    acc[0] += g.x * sp.x + g.y * sp.y;  acc[1] += g.y * sp.x - g.x * sp.y;
    acc[2] += g.x * sp.z + g.y * sp.w;  acc[3] += g.y * sp.z - g.x * sp.w;
    acc[4] += g.z * sp.x + g.w * sp.y;  acc[5] += g.w * sp.x - g.z * sp.y;
    acc[6] += g.z * sp.z + g.w * sp.w;  acc[7] += g.w * sp.z - g.z * sp.w;
  }
  static __device__ __forceinline__ void store_sums(const Grads&, double* part, size_t row, const double* acc) {
#pragma unroll
    for (int i = 0; i < kSums; ++i) part[row * kSums + i] = acc[i];
  }
};

// D-LinOSS (time-invariant parameters): the four variants' coefficient tables,
// adjoint and chain rule in double, as the reference's device kernels run them
// for complex128 (dlinoss_imex1_cuda.cu:23-172 and siblings):
//   new0 = c0 s0 + c1 s1 + c2 bu ;  new1 = c3 s0 + c4 s1 + c5 bu
// except imex1 (new1 = new0 + s1) and ex (new1 = c3 s0 + s1); tables
// dlinoss_imex1.cpp:32-48, dlinoss_imex2.cpp:35-47, dlinoss_im.cpp:34-50,
// dlinoss_ex.cpp:33-42.  No clamp on dt (the reference applies none).
// Adjoint: mu_t = carry + (0, grad_out_t); grad_bu_t = f^T mu_t; carry to
// t-1 = M^T mu_t (dlinoss_imex1.cpp:200-208, dlinoss_imex2.cpp:222-230,
// dlinoss_im.cpp:229-237, dlinoss_ex.cpp:189-197).
struct Coef64 {
  double c0, c1, c2, c3, c4, c5;
};

struct DlParams64 {
  const double* a;
  const double* g;
  const double* dt;
  int P;
};

template <int V>
struct Dl64 {
  static constexpr bool kVarying = false;
  // Sums per channel the chain rule reads (G_ij = sum <mu_i, s_j,t-1>, F_i =
  // sum <mu_i, bu_t>, real inner products of complex numbers), in the
  // combinations each variant needs:
  //   imex1: G00 + G10, G01 + G11, F0 + F1     ex: G00, G01, F0 + G10
  //   im:    G00, G01, G11, F0 + G10, F1       imex2: G00, G01, G10, G11, F0, F1
  static constexpr int kSums =
      (V == OSSM_DLINOSS_IMEX1 || V == OSSM_DLINOSS_EX) ? 3 : (V == OSSM_DLINOSS_IM ? 5 : 6);
  static constexpr Chunking kFwd{128, 10, 256 * kMb, 5}, kBwd{100, 8, 300 * kMb, 4};
  using Params = DlParams64;
  using Mat = RMatD;
  using Grads = NoGrads64;
  using In = double2;
  using Coef = Coef64;
  static __device__ __forceinline__ int width(const Params& prm) { return prm.P; }
  static __device__ __forceinline__ Coef coef(const Params& prm, int, int, int p) {
    const double alpha = prm.a[p], gamma = prm.g[p], sigma = prm.dt[p];
    if constexpr (V == OSSM_DLINOSS_IMEX1) {
      const double inv = 1.0 / (1.0 + sigma * gamma);
      const double s2i = sigma * sigma * inv;
      return {inv, -alpha * s2i, s2i, 0.0, 0.0, 0.0};
    } else if constexpr (V == OSSM_DLINOSS_IMEX2) {
      const double s2 = sigma * sigma;
      return {1.0 - sigma * gamma, -sigma * alpha, sigma, sigma - s2 * gamma, 1.0 - s2 * alpha, s2};
    } else if constexpr (V == OSSM_DLINOSS_IM) {
      const double s2 = sigma * sigma;
      const double inv = 1.0 / (1.0 + sigma * gamma + s2 * alpha);
      const double si = sigma * inv;
      return {inv, -alpha * si, si, si, (1.0 + sigma * gamma) * inv, s2 * inv};
    } else {
      return {1.0 - sigma * gamma, -sigma * alpha, sigma, sigma, 0.0, 0.0};
    }
  }
  static __device__ __forceinline__ In load_in(const double2* in, size_t e) { return in[e]; }
  static __device__ __forceinline__ St step(const Coef& k, St s, In b) {
    St n;
    n.x = s.x * k.c0 + s.z * k.c1 + b.x * k.c2;
    n.y = s.y * k.c0 + s.w * k.c1 + b.y * k.c2;
    if constexpr (V == OSSM_DLINOSS_IMEX1) {
      n.z = n.x + s.z;
      n.w = n.y + s.w;
    } else if constexpr (V == OSSM_DLINOSS_EX) {
      n.z = s.x * k.c3 + s.z;
      n.w = s.y * k.c3 + s.w;
    } else {
      n.z = s.x * k.c3 + s.z * k.c4 + b.x * k.c5;
      n.w = s.y * k.c3 + s.w * k.c4 + b.y * k.c5;
    }
    return n;
  }
  static __device__ __forceinline__ Mat matrix(const Coef& k) {
    if constexpr (V == OSSM_DLINOSS_IMEX1) return {k.c0, k.c1, k.c0, 1.0 + k.c1};
    else if constexpr (V == OSSM_DLINOSS_EX) return {k.c0, k.c1, k.c3, 1.0};
    else return {k.c0, k.c1, k.c3, k.c4};
  }
  static __device__ __forceinline__ St mu(St y, In go) { return {y.x, y.y, y.z + go.x, y.w + go.y}; }
  static __device__ __forceinline__ St rev(const Coef& k, St m) {
    if constexpr (V == OSSM_DLINOSS_IMEX1) {
      const double tr = m.x + m.z, ti = m.y + m.w;
      return {tr * k.c0, ti * k.c0, m.z + tr * k.c1, m.w + ti * k.c1};
    } else if constexpr (V == OSSM_DLINOSS_EX) {
      return {m.x * k.c0 + m.z * k.c3, m.y * k.c0 + m.w * k.c3, m.x * k.c1 + m.z, m.y * k.c1 + m.w};
    } else {
      return {m.x * k.c0 + m.z * k.c3, m.y * k.c0 + m.w * k.c3, m.x * k.c1 + m.z * k.c4,
              m.y * k.c1 + m.w * k.c4};
    }
  }
  static __device__ __forceinline__ void grads(const Coef& k, St m, St sp, In b, double2* gin, size_t e,
                                               double* acc, const Grads&) {
    if constexpr (V == OSSM_DLINOSS_IMEX1) {
      const double tr = m.x + m.z, ti = m.y + m.w;
      acc[0] += tr * sp.x + ti * sp.y;
      acc[1] += tr * sp.z + ti * sp.w;
      acc[2] += tr * b.x + ti * b.y;
      stream_store(gin + e, make_double2(tr * k.c2, ti * k.c2));
    } else if constexpr (V == OSSM_DLINOSS_EX) {
      acc[0] += m.x * sp.x + m.y * sp.y;
      acc[1] += m.x * sp.z + m.y * sp.w;
      acc[2] += m.x * b.x + m.y * b.y + m.z * sp.x + m.w * sp.y;
      stream_store(gin + e, make_double2(m.x * k.c2, m.y * k.c2));
    } else {
      if constexpr (V == OSSM_DLINOSS_IM) {
        acc[0] += m.x * sp.x + m.y * sp.y;
        acc[1] += m.x * sp.z + m.y * sp.w;
        acc[2] += m.z * sp.z + m.w * sp.w;
        acc[3] += m.x * b.x + m.y * b.y + m.z * sp.x + m.w * sp.y;
        acc[4] += m.z * b.x + m.w * b.y;
      } else {
        acc[0] += m.x * sp.x + m.y * sp.y;
        acc[1] += m.x * sp.z + m.y * sp.w;
        acc[2] += m.z * sp.x + m.w * sp.y;
        acc[3] += m.z * sp.z + m.w * sp.w;
        acc[4] += m.x * b.x + m.y * b.y;
        acc[5] += m.z * b.x + m.w * b.y;
      }
      stream_store(gin + e, make_double2(m.x * k.c2 + m.z * k.c5, m.y * k.c2 + m.w * k.c5));
    }
  }
  static __device__ __forceinline__ void store_sums(const Grads&, double* part, size_t row, const double* acc) {
#pragma unroll
    for (int i = 0; i < kSums; ++i) part[row * kSums + i] = acc[i];
  }
};

// ---- the chunked scans --------------------------------------------------------
// One wave per (64 channels, chunk): blockIdx.x = channel group, blockIdx.y =
// chunk of CL steps.  agg[chunk nc + ch]: where the chunk ends from a zero carry
// (two double2); tr[chunk nc + ch]: the product of its transitions (kVarying).
struct Plan64 {
  int L, nc, CL, n_chunks;
  double2* agg;
  RMatD* tr;
};

// Whether every component is finite (x - x is 0, or NaN for infinities and NaN).
__device__ __forceinline__ bool st_finite(St s) {
  return (s.x - s.x) + (s.y - s.y) + (s.z - s.z) + (s.w - s.w) == 0.0;
}

template <class M>
__global__ __launch_bounds__(kWave) void chunk64_fwd_kernel(typename M::Params prm,
                                                            const double2* __restrict__ in, Plan64 pl) {
  const int ch = static_cast<int>(blockIdx.x) * kWave + static_cast<int>(threadIdx.x);
  if (ch >= pl.nc) return;
  const int c = static_cast<int>(blockIdx.y), t0 = c * pl.CL;  // the last chunk is not launched: full
  const int m = ch % M::width(prm);
  auto k = M::coef(prm, t0, ch, m);
  St s = st_zero();
  RMatD P{1.0, 0.0, 0.0, 1.0};
#pragma unroll 8
  for (int t = t0; t < t0 + pl.CL; ++t) {
    if constexpr (M::kVarying) k = M::coef(prm, t, ch, m);
    s = M::step(k, s, M::load_in(in, static_cast<size_t>(t) * pl.nc + ch));
    if constexpr (M::kVarying) P = mat_mul(M::matrix(k), P);
  }
  const size_t row = static_cast<size_t>(c) * pl.nc + ch;
  store_st(pl.agg + 2 * row, s);
  if constexpr (M::kVarying) pl.tr[row] = P;
}

template <class M>
__global__ __launch_bounds__(kWave) void scan64_fwd_kernel(typename M::Params prm,
                                                           const double2* __restrict__ in,
                                                           double2* __restrict__ states, Plan64 pl) {
  const int ch = static_cast<int>(blockIdx.x) * kWave + static_cast<int>(threadIdx.x);
  if (ch >= pl.nc) return;
  const int c = static_cast<int>(blockIdx.y);
  const int t0 = c * pl.CL, t1 = min(pl.L, t0 + pl.CL);
  const int m = ch % M::width(prm);
  auto k = M::coef(prm, t0, ch, m);
  St s = st_zero();
  if (c > 0) {
    if constexpr (M::kVarying) {
#pragma unroll 4
      for (int j = 0; j < c; ++j) {
        const size_t row = static_cast<size_t>(j) * pl.nc + ch;
        s = st_add(st_apply(pl.tr[row], s), load_st(pl.agg + 2 * row));
      }
    } else {
      const auto MC = pow64(M::matrix(k), pl.CL);
#pragma unroll 8
      for (int j = 0; j < c; ++j)
        s = st_add(st_apply(MC, s), load_st(pl.agg + 2 * (static_cast<size_t>(j) * pl.nc + ch)));
    }
    // A chunk's transition may overflow where no state does (times zero: NaN), and an
    // infinite state goes on step by step in its own way: walk the steps before the
    // chunk instead, which takes what one lane per sequence took.
    if (!st_finite(s)) {
      s = st_zero();
#pragma unroll 4
      for (int t = 0; t < t0; ++t) {
        if constexpr (M::kVarying) k = M::coef(prm, t, ch, m);
        s = M::step(k, s, M::load_in(in, static_cast<size_t>(t) * pl.nc + ch));
      }
    }
  }
#pragma unroll 8
  for (int t = t0; t < t1; ++t) {
    const size_t e = static_cast<size_t>(t) * pl.nc + ch;
    if constexpr (M::kVarying) k = M::coef(prm, t, ch, m);
    s = M::step(k, s, M::load_in(in, e));
    store_st(states + 2 * e, s);
  }
}

// Reverse: chunk blockIdx.y + 1 (the first chunk's aggregate is not needed).
template <class M>
__global__ __launch_bounds__(kWave) void chunk64_bwd_kernel(typename M::Params prm,
                                                            const double2* __restrict__ gout, Plan64 pl) {
  const int ch = static_cast<int>(blockIdx.x) * kWave + static_cast<int>(threadIdx.x);
  if (ch >= pl.nc) return;
  const int c = static_cast<int>(blockIdx.y) + 1;
  const int t0 = c * pl.CL, t1 = min(pl.L, t0 + pl.CL);
  const int m = ch % M::width(prm);
  auto k = M::coef(prm, t0, ch, m);
  St y = st_zero();
  RMatD P{1.0, 0.0, 0.0, 1.0};
#pragma unroll 8
  for (int t = t1 - 1; t >= t0; --t) {
    if constexpr (M::kVarying) k = M::coef(prm, t, ch, m);
    y = M::rev(k, M::mu(y, M::load_in(gout, static_cast<size_t>(t) * pl.nc + ch)));
    if constexpr (M::kVarying) P = mat_mul(adjoint64(M::matrix(k)), P);
  }
  const size_t row = static_cast<size_t>(c) * pl.nc + ch;
  store_st(pl.agg + 2 * row, y);
  if constexpr (M::kVarying) pl.tr[row] = P;
}

template <class M>
__global__ __launch_bounds__(kWave) void scan64_bwd_kernel(
    typename M::Params prm, const double2* __restrict__ in, const double2* __restrict__ states,
    const double2* __restrict__ gout, double2* __restrict__ gin, typename M::Grads dst,
    double* __restrict__ part, Plan64 pl) {
  const int ch = static_cast<int>(blockIdx.x) * kWave + static_cast<int>(threadIdx.x);
  if (ch >= pl.nc) return;
  const int c = static_cast<int>(blockIdx.y);
  const int t0 = c * pl.CL, t1 = min(pl.L, t0 + pl.CL);
  const int m = ch % M::width(prm);
  auto k = M::coef(prm, t0, ch, m);
  St y = st_zero();
  if (c + 1 < pl.n_chunks) {
    if constexpr (M::kVarying) {
#pragma unroll 4
      for (int j = pl.n_chunks - 1; j > c; --j) {
        const size_t row = static_cast<size_t>(j) * pl.nc + ch;
        y = st_add(st_apply(pl.tr[row], y), load_st(pl.agg + 2 * row));
      }
    } else {
      // the last chunk may be short, but nothing enters it: its power never matters
      const auto MC = pow64(adjoint64(M::matrix(k)), pl.CL);
#pragma unroll 8
      for (int j = pl.n_chunks - 1; j > c; --j)
        y = st_add(st_apply(MC, y), load_st(pl.agg + 2 * (static_cast<size_t>(j) * pl.nc + ch)));
    }
    if (!st_finite(y)) {  // as in scan64_fwd_kernel
      y = st_zero();
#pragma unroll 4
      for (int t = pl.L - 1; t >= t1; --t) {
        if constexpr (M::kVarying) k = M::coef(prm, t, ch, m);
        y = M::rev(k, M::mu(y, M::load_in(gout, static_cast<size_t>(t) * pl.nc + ch)));
      }
    }
  }
  double acc[M::kSums];
#pragma unroll
  for (int i = 0; i < M::kSums; ++i) acc[i] = 0.0;
#pragma unroll 4
  for (int t = t1 - 1; t >= t0; --t) {
    const size_t e = static_cast<size_t>(t) * pl.nc + ch;
    if constexpr (M::kVarying) k = M::coef(prm, t, ch, m);
    const St g = M::mu(y, M::load_in(gout, e));
    // s_{t-1}, zero before the first step
    St sp = load_st(states + 2 * (t > 0 ? e - pl.nc : e));
    if (t == 0) sp = st_zero();
    typename M::In b{};
    if (in != nullptr) b = M::load_in(in, e);
    M::grads(k, g, sp, b, gin, e, acc, dst);
    y = M::rev(k, g);
  }
  M::store_sums(dst, part, static_cast<size_t>(c) * pl.nc + ch, acc);
}

// ---- sums over rows -------------------------------------------------------------
// out[n C + c] = sum_{r < R} in[(n R + r) C + c], one workgroup per (n, 16 columns):
// 16 columns by 16 row lanes (a lane adds rows rl, rl + 16, ... in order, then
// the 16 partial sums are added in order).  One lane per column walking all R
// rows took as long as the scan once R counts the chunks.
constexpr int kSumCols = 16, kSumRows = kBlock64 / kSumCols;

__global__ __launch_bounds__(kBlock64) void rows_sum64_kernel(const double* __restrict__ in,
                                                              double* __restrict__ out, int R, int C) {
  __shared__ double s_p[kSumRows][kSumCols];
  const int cl = static_cast<int>(threadIdx.x) % kSumCols, rl = static_cast<int>(threadIdx.x) / kSumCols;
  const int n_cb = (C + kSumCols - 1) / kSumCols;
  const size_t n = blockIdx.x / n_cb;
  const int c = static_cast<int>(blockIdx.x % n_cb) * kSumCols + cl;
  double s = 0.0;
  if (c < C) {
    const double* src = in + n * R * C + c;
#pragma unroll 4
    for (int r = rl; r < R; r += kSumRows) s += src[static_cast<size_t>(r) * C];
  }
  s_p[rl][cl] = s;
  __syncthreads();
  if (rl == 0 && c < C) {
#pragma unroll
    for (int v = 1; v < kSumRows; ++v) s += s_p[v][cl];
    out[n * C + c] = s;
  }
}

__global__ __launch_bounds__(kBlock64) void sdl64_zero_kernel(double* __restrict__ p, long long n) {
  const long long i = static_cast<long long>(blockIdx.x) * kBlock64 + threadIdx.x;
  if (i < n) p[i] = 0.0;
}

// D-LinOSS: the (chunk, batch row) sums of each oscillator added in a fixed
// order (as rows_sum64_kernel), then the chain rule to (a, g, dt): imex1
// dlinoss_imex1.cpp:219-232, im dlinoss_im.cpp:236-263, imex2 / ex by
// differentiating the coefficient tables (the terms the reference accumulates
// per step).
template <int V>
__global__ __launch_bounds__(kBlock64) void dl64_param_kernel(DlParams64 prm,
                                                              const double* __restrict__ part,
                                                              double* __restrict__ grad_a,
                                                              double* __restrict__ grad_g,
                                                              double* __restrict__ grad_step,
                                                              int R) {
  constexpr int NS = Dl64<V>::kSums;
  __shared__ double s_p[kSumRows][kSumCols][NS];
  const int cl = static_cast<int>(threadIdx.x) % kSumCols, rl = static_cast<int>(threadIdx.x) / kSumCols;
  const int p = static_cast<int>(blockIdx.x) * kSumCols + cl;
  double S[NS];
#pragma unroll
  for (int i = 0; i < NS; ++i) S[i] = 0.0;
  if (p < prm.P) {
#pragma unroll 2
    for (int r = rl; r < R; r += kSumRows) {
      const double* src = part + (static_cast<size_t>(r) * prm.P + p) * NS;
#pragma unroll
      for (int i = 0; i < NS; ++i) S[i] += src[i];
    }
  }
#pragma unroll
  for (int i = 0; i < NS; ++i) s_p[rl][cl][i] = S[i];
  __syncthreads();
  if (rl != 0 || p >= prm.P) return;
  for (int v = 1; v < kSumRows; ++v)
#pragma unroll
    for (int i = 0; i < NS; ++i) S[i] += s_p[v][cl][i];
  const double a = prm.a[p], g = prm.g[p], dt = prm.dt[p];
  double ga, gg, gs;
  if constexpr (V == OSSM_DLINOSS_IMEX1) {
    const double inv = 1.0 / (1.0 + dt * g);
    const double s2i = dt * dt * inv;
    const double gs2i = S[2] - a * S[1];
    ga = -s2i * S[1];
    const double inv_total = S[0] + gs2i * dt * dt;
    gs = gs2i * (2.0 * dt * inv) - inv_total * g * inv * inv;
    gg = -inv_total * dt * inv * inv;
  } else if constexpr (V == OSSM_DLINOSS_IMEX2) {
    ga = -dt * S[1] - dt * dt * S[3];
    gg = -dt * S[0] - dt * dt * S[2];
    gs = -g * S[0] - a * S[1] + (1.0 - 2.0 * dt * g) * S[2] - 2.0 * dt * a * S[3] + S[4] +
         2.0 * dt * S[5];
  } else if constexpr (V == OSSM_DLINOSS_IM) {
    const double inv = 1.0 / (1.0 + dt * g + dt * dt * a);
    const double si = dt * inv;
    const double gsi = S[3] - a * S[1];
    double ginv = S[0] + S[2] * (1.0 + dt * g);
    const double gt = S[2] * inv;
    ga = -si * S[1];
    gg = gt * dt;
    gs = gt * g + gsi * inv + S[4] * (2.0 * dt * inv);
    ginv += gsi * dt + S[4] * dt * dt;
    const double gden = -ginv * inv * inv;
    ga += gden * dt * dt;
    gg += gden * dt;
    gs += gden * (g + 2.0 * dt * a);
  } else {
    ga = -dt * S[1];
    gg = -dt * S[0];
    gs = -g * S[0] - a * S[1] + S[2];
  }
  grad_a[p] = ga;
  grad_g[p] = gg;
  grad_step[p] = gs;
}

unsigned blocks_for(long long n) { return static_cast<unsigned>((n + kBlock64 - 1) / kBlock64); }

struct Shape64 {
  const double* p;
  int64_t la, ba;
};

int check64(int variant, const Shape64 (&s)[3], int64_t L, int64_t B, int64_t M, const char* what) {
  if (variant < 0 || variant > 3)
    return set_error(OSSM_ERR_INVALID_ARGUMENT, "Unknown selective D-LinOSS variant code");
  if (L < 0 || B < 0 || M < 0)
    return set_error(OSSM_ERR_INVALID_ARGUMENT, std::string(what) + ": negative size");
  if (L > INT_MAX / 2 || B * M > INT_MAX / 2 || L * B * M > (int64_t(1) << 40))
    return set_error(OSSM_ERR_UNSUPPORTED, std::string(what) + ": size exceeds 32-bit indexing");
  const char* names[3] = {"A", "G", "step"};
  for (int p = 0; p < 3; ++p) {
    if (s[p].p == nullptr)
      return set_error(OSSM_ERR_INVALID_ARGUMENT, std::string(what) + ": null " + names[p]);
    if (!(s[p].la == 1 || s[p].la == L) || !(s[p].ba == 1 || s[p].ba == B))
      return set_error(OSSM_ERR_INVALID_ARGUMENT, std::string(names[p]) +
                                                      " must have shape (L,B,M) with optional singleton L/B axes");
  }
  return OSSM_OK;
}

Params64 params64(const Shape64 (&s)[3], int64_t L, int64_t B, int64_t M) {
  Params64 prm{};
  for (int p = 0; p < 3; ++p) {
    prm.v[p].p = s[p].p;
    prm.v[p].t_stride = (s[p].la == 1 && L > 1) ? 0 : s[p].ba * M;
    prm.v[p].by_channel = s[p].ba == B ? 1 : 0;
  }
  prm.M = static_cast<int>(M);
  return prm;
}

}  // namespace
}  // namespace ossm

namespace ossm {
namespace {

// Chunks per sequence: sqrt(L), which balances a lane's own steps against the
// aggregates it folds (up to as many as there are chunks), and no more waves
// than 2048 (two per SIMD, 64 channels each): beyond that the second read
// of the inputs costs more than the waves hide.  Swept over factors 0.7 to 2.8
// of sqrt(L) and 2048 to 8192 waves at seven shapes: within 7 % of the best at
// each.  One lane per sequence against this plan, D-LinOSS imex2 forward /
// backward, us, [L, B, P]: [2048, 8, 128] 360 / 820 -> 31 / 38 (4.4 TB/s of the
// backward's 80 B per state-step); [512, 64, 256] 217 / 362 -> 104 / 112;
// [4096, 32, 128] 1256 / 2584 -> 234 / 267; [16384, 4, 128] 4896 / 10137 -> 121 / 130.
// One chunk -> the plan at the lines drawn, groups of 64 channels (their chunks):
//   forward, L = 100  1 group      D-LinOSS 10 -> 12  LinOSS 12 -> 12  selective 22 -> 13
//            L = 300  256 (8)               47 -> 50         113 -> 80          169 -> 111
//            L = 1500 400 (5)              558 -> 498        703 -> 663         955 -> 941
//                     512 (4)              561 -> 601        744 -> 806         983 -> 1160
//                     1024 (2)             967 -> 1120      1281 -> 1534       1402 -> 2234
//   backward, L = 49  1 group               17 -> 19          15 -> 17           25 -> 21
//            L = 144  256 (8)               43 -> 41          42 -> 54           97 -> 61
//            L = 1500 340 (6)              718 -> 463        708 -> 734        1564 -> 1006
//                     512 (4)              764 -> 683        875 -> 1053       1640 -> 1494
//                     680 (3)              876 -> 885       1198 -> 1410       1771 -> 1960
//            (680, parameters constant over time)                             1460 -> 1269
int chunks64(int64_t L, int64_t nc, const Chunking& c, int64_t bytes) {
  const int64_t groups = (nc + kWave - 1) / kWave, cap = 2048 / groups;
  const int64_t n = std::min<int64_t>(cap, static_cast<int64_t>(std::sqrt(static_cast<double>(L))));
  if (n < 2 || L < c.min_len || cap < (bytes >= c.big ? c.min_chunks_big : c.min_chunks)) return 1;
  const int64_t cl = (L + n - 1) / n;
  return static_cast<int>((L + cl - 1) / cl);
}

// The chunk plan of a call that moves `bytes` bytes and the workspace it lives in:
// `sums(n_chunks)` doubles for the caller's partial sums, then the aggregates and (varying) the transition
// products.  When the workspace cannot be had (under stream capture it may not
// grow; a full device) the call runs as one chunk, which needs only the sums.
template <class Sums>
int plan64(StreamCall& call, int64_t L, int64_t nc, bool varying, const Chunking& cut, int64_t bytes, Sums sums,
           Plan64* pl, double** part) {
  // a captured call without sums takes no workspace, so that its graph may replay
  // beside the capture stream's own work
  int n = call.capturing() && sums(1) == 0 ? 1 : chunks64(L, nc, cut, bytes);
  for (;;) {
    const size_t rows = n > 1 ? static_cast<size_t>(n) * nc : 0;
    const size_t n_sums = (sums(n) + 1) & ~size_t(1);  // 16-byte aligned double2 behind them
    const size_t bytes = n_sums * sizeof(double) + rows * (2 * sizeof(double2) + (varying ? sizeof(RMatD) : 0));
    void* raw = nullptr;
    if (bytes > 0) {
      if (int rc = acquire_workspace(call, bytes, &raw)) {
        if (n == 1) return rc;
        (void)hipGetLastError();
        clear_error();
        n = 1;
        continue;
      }
    }
    auto* base = static_cast<double*>(raw);
    pl->L = static_cast<int>(L);
    pl->nc = static_cast<int>(nc);
    pl->n_chunks = n;
    pl->CL = static_cast<int>((L + n - 1) / n);
    *part = base;
    pl->agg = rows ? reinterpret_cast<double2*>(base + n_sums) : nullptr;
    pl->tr = rows && varying ? reinterpret_cast<RMatD*>(pl->agg + 2 * rows) : nullptr;
    return OSSM_OK;
  }
}

// step_bytes: read and written per state-step, once each
template <class M>
int run_forward64(const typename M::Params& prm, const void* in, void* states, int64_t L, int64_t nc,
                  int64_t step_bytes, hipStream_t stream) {
  StreamCall call(stream);
  if (call.status()) return call.status();
  Plan64 pl{};
  double* part = nullptr;
  if (int rc = plan64(call, L, nc, M::kVarying, M::kFwd, L * nc * step_bytes, [](int) { return size_t(0); }, &pl,
                      &part))
    return rc;
  const unsigned groups = static_cast<unsigned>((nc + kWave - 1) / kWave);
  const auto* src = static_cast<const double2*>(in);
  if (pl.n_chunks > 1) {
    hipLaunchKernelGGL(chunk64_fwd_kernel<M>, dim3(groups, pl.n_chunks - 1), dim3(kWave), 0, stream, prm,
                       src, pl);
    if (int rc = launch_check("chunk64_fwd_kernel")) return rc;
  }
  hipLaunchKernelGGL(scan64_fwd_kernel<M>, dim3(groups, pl.n_chunks), dim3(kWave), 0, stream, prm, src,
                     static_cast<double2*>(states), pl);
  return launch_check("scan64_fwd_kernel");
}

template <class M>
int run_backward64(const typename M::Params& prm, const void* in, const void* states, const void* gout,
                   void* gin, const typename M::Grads& dst, double* part, const Plan64& pl,
                   hipStream_t stream) {
  const unsigned groups = static_cast<unsigned>((pl.nc + kWave - 1) / kWave);
  const auto* go = static_cast<const double2*>(gout);
  if (pl.n_chunks > 1) {
    hipLaunchKernelGGL(chunk64_bwd_kernel<M>, dim3(groups, pl.n_chunks - 1), dim3(kWave), 0, stream, prm,
                       go, pl);
    if (int rc = launch_check("chunk64_bwd_kernel")) return rc;
  }
  hipLaunchKernelGGL(scan64_bwd_kernel<M>, dim3(groups, pl.n_chunks), dim3(kWave), 0, stream, prm,
                     static_cast<const double2*>(in), static_cast<const double2*>(states), go,
                     static_cast<double2*>(gin), dst, part, pl);
  return launch_check("scan64_bwd_kernel");
}

int rows_sum64(const double* in, double* out, int64_t n, int64_t R, int64_t C, hipStream_t stream) {
  const int64_t blocks = n * ((C + kSumCols - 1) / kSumCols);
  if (blocks > INT_MAX || R > INT_MAX)
    return set_error(OSSM_ERR_UNSUPPORTED, "rows_sum64: problem too large for one launch grid");
  hipLaunchKernelGGL(rows_sum64_kernel, dim3(static_cast<unsigned>(blocks)), dim3(kBlock64), 0, stream, in,
                     out, static_cast<int>(R), static_cast<int>(C));
  return launch_check("rows_sum64_kernel");
}

}  // namespace
}  // namespace ossm

using namespace ossm;

extern "C" {

int ossm_sdlinoss_forward_f64(int variant, const double* A, int64_t a_len, int64_t a_batch,
                              const double* G, int64_t g_len, int64_t g_batch, const double* step,
                              int64_t s_len, int64_t s_batch, const void* bu, void* states,
                              int64_t length, int64_t batch, int64_t ssm, ossm_stream_t stream_v) {
  clear_error();
  const Shape64 shapes[3] = {{A, a_len, a_batch}, {G, g_len, g_batch}, {step, s_len, s_batch}};
  if (length == 0 || batch == 0 || ssm == 0) {
    if (variant < 0 || variant > 3)
      return set_error(OSSM_ERR_INVALID_ARGUMENT, "Unknown selective D-LinOSS variant code");
    return OSSM_OK;
  }
  if (int rc = check64(variant, shapes, length, batch, ssm, "sdlinoss_forward_f64")) return rc;
  if (!bu || !states) return set_error(OSSM_ERR_INVALID_ARGUMENT, "sdlinoss_forward_f64: null pointer");
  const Params64 prm = params64(shapes, length, batch, ssm);
  int64_t step_bytes = 48;  // bu and the states, and each parameter that is full size
  for (const Shape64& s : shapes) step_bytes += s.la == length && s.ba == batch ? 8 : 0;
  hipStream_t stream = static_cast<hipStream_t>(stream_v);
  switch (variant) {
    case OSSM_DLINOSS_IMEX1:
      return run_forward64<Sdl64<OSSM_DLINOSS_IMEX1>>(prm, bu, states, length, batch * ssm, step_bytes, stream);
    case OSSM_DLINOSS_IMEX2:
      return run_forward64<Sdl64<OSSM_DLINOSS_IMEX2>>(prm, bu, states, length, batch * ssm, step_bytes, stream);
    case OSSM_DLINOSS_IM:
      return run_forward64<Sdl64<OSSM_DLINOSS_IM>>(prm, bu, states, length, batch * ssm, step_bytes, stream);
    default:
      return run_forward64<Sdl64<OSSM_DLINOSS_EX>>(prm, bu, states, length, batch * ssm, step_bytes, stream);
  }
}

int ossm_sdlinoss_backward_f64(int variant, const double* A, int64_t a_len, int64_t a_batch,
                               const double* G, int64_t g_len, int64_t g_batch,
                               const double* step, int64_t s_len, int64_t s_batch, const void* bu,
                               const void* states, const void* grad_output, double* grad_A,
                               double* grad_G, double* grad_step, void* grad_bu, int64_t length,
                               int64_t batch, int64_t ssm, ossm_stream_t stream_v) {
  clear_error();
  hipStream_t stream = static_cast<hipStream_t>(stream_v);
  StreamCall call(stream);
  if (call.status()) return call.status();
  const Shape64 shapes[3] = {{A, a_len, a_batch}, {G, g_len, g_batch}, {step, s_len, s_batch}};
  double* const grads[3] = {grad_A, grad_G, grad_step};
  if (length == 0 || batch == 0 || ssm == 0) {
    if (variant < 0 || variant > 3)
      return set_error(OSSM_ERR_INVALID_ARGUMENT, "Unknown selective D-LinOSS variant code");
    // nothing to scan: zero parameter gradients (the reference's zeros_like)
    for (int p = 0; p < 3; ++p) {
      if (grads[p] == nullptr)
        return set_error(OSSM_ERR_INVALID_ARGUMENT, "sdlinoss_backward_f64: null pointer");
      const long long n = shapes[p].la * shapes[p].ba * ssm;
      if (n <= 0) continue;
      hipLaunchKernelGGL(sdl64_zero_kernel, dim3(blocks_for(n)), dim3(kBlock64), 0, stream,
                         grads[p], n);
      if (int rc = launch_check("sdl64_zero_kernel")) return rc;
    }
    return OSSM_OK;
  }
  if (int rc = check64(variant, shapes, length, batch, ssm, "sdlinoss_backward_f64")) return rc;
  if (!bu || !states || !grad_output || !grad_A || !grad_G || !grad_step || !grad_bu)
    return set_error(OSSM_ERR_INVALID_ARGUMENT, "sdlinoss_backward_f64: null pointer");
  const Params64 prm = params64(shapes, length, batch, ssm);
  const int64_t nc = batch * ssm;

  // Gradients that are summed go through the workspace first: [L, B, M] per
  // element (broadcast over batch only), or [n_chunks, B, M] time sums
  // (broadcast over time, or over both).
  Grads64 dst{};
  bool rt[3], rb[3];
  for (int p = 0; p < 3; ++p) {
    rt[p] = shapes[p].la == 1 && length > 1;
    rb[p] = shapes[p].ba == 1 && batch > 1;
    dst.mode[p] = rt[p] ? 1 : (rb[p] ? 2 : 0);
  }
  auto rows_of = [&](int p, int n) -> size_t {
    if (rt[p]) return n > 1 || rb[p] ? static_cast<size_t>(n) * nc : 0;
    return rb[p] ? static_cast<size_t>(length) * nc : 0;
  };
  Plan64 pl{};
  double* ws = nullptr;
  using Any = Sdl64<OSSM_DLINOSS_IMEX1>;
  const bool constant = rt[0] && rt[1] && rt[2];  // over time: no gradient per step
  if (int rc = plan64(call, length, nc, true, constant ? Any::kBwdConstant : Any::kBwd, 0,
                      [&](int n) { return rows_of(0, n) + rows_of(1, n) + rows_of(2, n); }, &pl, &ws))
    return rc;
  for (int p = 0; p < 3; ++p) {
    const size_t rows = rows_of(p, pl.n_chunks);
    dst.out[p] = rows ? ws : grads[p];
    ws += rows;
  }
  int rc = OSSM_OK;
  switch (variant) {
    case OSSM_DLINOSS_IMEX1:
      rc = run_backward64<Sdl64<OSSM_DLINOSS_IMEX1>>(prm, bu, states, grad_output, grad_bu, dst, nullptr, pl, stream);
      break;
    case OSSM_DLINOSS_IMEX2:
      rc = run_backward64<Sdl64<OSSM_DLINOSS_IMEX2>>(prm, bu, states, grad_output, grad_bu, dst, nullptr, pl, stream);
      break;
    case OSSM_DLINOSS_IM:
      rc = run_backward64<Sdl64<OSSM_DLINOSS_IM>>(prm, bu, states, grad_output, grad_bu, dst, nullptr, pl, stream);
      break;
    default:
      rc = run_backward64<Sdl64<OSSM_DLINOSS_EX>>(prm, bu, states, grad_output, grad_bu, dst, nullptr, pl, stream);
  }
  if (rc) return rc;
  for (int p = 0; p < 3; ++p) {
    if (dst.out[p] == grads[p]) continue;
    if (rt[p])  // [n_chunks][B][M] over the chunks, and over the batch rows when shared by them
      rc = rb[p] ? rows_sum64(dst.out[p], grads[p], 1, int64_t(pl.n_chunks) * batch, ssm, stream)
                 : rows_sum64(dst.out[p], grads[p], 1, pl.n_chunks, nc, stream);
    else  // [L][B][M] over the batch rows
      rc = rows_sum64(dst.out[p], grads[p], length, batch, ssm, stream);
    if (rc) return rc;
  }
  return OSSM_OK;
}

int ossm_linoss_forward_f64(const void* m11, const void* m12, const void* m21, const void* m22,
                            const void* b_seq, void* states, int64_t length, int64_t batch,
                            int64_t ssm, ossm_stream_t stream_v) {
  clear_error();
  if (length < 0 || batch < 0 || ssm < 0)
    return set_error(OSSM_ERR_INVALID_ARGUMENT, "linoss_forward_f64: negative size");
  if (length == 0 || batch == 0 || ssm == 0) return OSSM_OK;
  if (length > INT_MAX / 2 || batch * ssm > INT_MAX / 2 || length * batch * ssm > (int64_t(1) << 40))
    return set_error(OSSM_ERR_UNSUPPORTED, "linoss_forward_f64: size exceeds 32-bit indexing");
  if (!m11 || !m12 || !m21 || !m22 || !b_seq || !states)
    return set_error(OSSM_ERR_INVALID_ARGUMENT, "linoss_forward_f64: null pointer");
  const Lin64Params mp{{static_cast<const double2*>(m11), static_cast<const double2*>(m12),
                        static_cast<const double2*>(m21), static_cast<const double2*>(m22)},
                       static_cast<int>(ssm)};
  return run_forward64<Lin64>(mp, b_seq, states, length, batch * ssm, 64, static_cast<hipStream_t>(stream_v));
}

int ossm_linoss_backward_f64(const void* m11, const void* m12, const void* m21, const void* m22,
                             const void* states, const void* grad_output, void* grad_m,
                             void* grad_b, int64_t length, int64_t batch, int64_t ssm,
                             ossm_stream_t stream_v) {
  clear_error();
  hipStream_t stream = static_cast<hipStream_t>(stream_v);
  StreamCall call(stream);
  if (call.status()) return call.status();
  if (length < 0 || batch < 0 || ssm < 0)
    return set_error(OSSM_ERR_INVALID_ARGUMENT, "linoss_backward_f64: negative size");
  if (length > INT_MAX / 2 || batch * ssm > INT_MAX / 2 || length * batch * ssm > (int64_t(1) << 40))
    return set_error(OSSM_ERR_UNSUPPORTED, "linoss_backward_f64: size exceeds 32-bit indexing");
  if (!grad_m) return set_error(OSSM_ERR_INVALID_ARGUMENT, "linoss_backward_f64: null pointer");
  const long long n_m = 8 * ssm;  // [P, 2, 2] complex128 as doubles
  if (length == 0 || batch == 0 || ssm == 0) {
    if (n_m > 0) {
      hipLaunchKernelGGL(sdl64_zero_kernel, dim3(blocks_for(n_m)), dim3(kBlock64), 0, stream,
                         static_cast<double*>(grad_m), n_m);
      return launch_check("sdl64_zero_kernel");
    }
    return OSSM_OK;
  }
  if (!m11 || !m12 || !m21 || !m22 || !states || !grad_output || !grad_b)
    return set_error(OSSM_ERR_INVALID_ARGUMENT, "linoss_backward_f64: null pointer");
  const Lin64Params mp{{static_cast<const double2*>(m11), static_cast<const double2*>(m12),
                        static_cast<const double2*>(m21), static_cast<const double2*>(m22)},
                       static_cast<int>(ssm)};
  const int64_t nc = batch * ssm;
  Plan64 pl{};
  double* part = nullptr;
  if (int rc = plan64(call, length, nc, false, Lin64::kBwd, length * nc * 96,
                      [&](int n) { return static_cast<size_t>(n) * nc * Lin64::kSums; }, &pl, &part))
    return rc;
  if (int rc = run_backward64<Lin64>(mp, nullptr, states, grad_output, grad_b, NoGrads64{}, part, pl, stream))
    return rc;
  // [n_chunks B rows][P * 8 doubles]
  return rows_sum64(part, static_cast<double*>(grad_m), 1, int64_t(pl.n_chunks) * batch, n_m, stream);
}

int ossm_dlinoss_forward_f64(int variant, const double* a_diag, const double* g_diag,
                             const double* step, const void* bu, void* states, int64_t length,
                             int64_t batch, int64_t ssm, ossm_stream_t stream_v) {
  clear_error();
  if (variant < OSSM_DLINOSS_IMEX1 || variant > OSSM_DLINOSS_EX)
    return set_error(OSSM_ERR_INVALID_ARGUMENT, "Unknown D-LinOSS variant code");
  if (length < 0 || batch < 0 || ssm < 0)
    return set_error(OSSM_ERR_INVALID_ARGUMENT, "dlinoss_forward_f64: negative size");
  if (length == 0 || batch == 0 || ssm == 0) return OSSM_OK;
  if (length > INT_MAX / 2 || batch * ssm > INT_MAX / 2 || length * batch * ssm > (int64_t(1) << 40))
    return set_error(OSSM_ERR_UNSUPPORTED, "dlinoss_forward_f64: size exceeds 32-bit indexing");
  if (!a_diag || !g_diag || !step || !bu || !states)
    return set_error(OSSM_ERR_INVALID_ARGUMENT, "dlinoss_forward_f64: null pointer");
  const DlParams64 prm{a_diag, g_diag, step, static_cast<int>(ssm)};
  const int64_t nc = batch * ssm;
  hipStream_t stream = static_cast<hipStream_t>(stream_v);
  switch (variant) {
    case OSSM_DLINOSS_IMEX1: return run_forward64<Dl64<OSSM_DLINOSS_IMEX1>>(prm, bu, states, length, nc, 48, stream);
    case OSSM_DLINOSS_IMEX2: return run_forward64<Dl64<OSSM_DLINOSS_IMEX2>>(prm, bu, states, length, nc, 48, stream);
    case OSSM_DLINOSS_IM: return run_forward64<Dl64<OSSM_DLINOSS_IM>>(prm, bu, states, length, nc, 48, stream);
    default: return run_forward64<Dl64<OSSM_DLINOSS_EX>>(prm, bu, states, length, nc, 48, stream);
  }
}

int ossm_dlinoss_backward_f64(int variant, const double* a_diag, const double* g_diag,
                              const double* step, const void* bu, const void* states,
                              const void* grad_output, double* grad_a, double* grad_g,
                              double* grad_step, void* grad_bu, int64_t length, int64_t batch,
                              int64_t ssm, ossm_stream_t stream_v) {
  clear_error();
  hipStream_t stream = static_cast<hipStream_t>(stream_v);
  StreamCall call(stream);
  if (call.status()) return call.status();
  if (variant < OSSM_DLINOSS_IMEX1 || variant > OSSM_DLINOSS_EX)
    return set_error(OSSM_ERR_INVALID_ARGUMENT, "Unknown D-LinOSS variant code");
  if (length < 0 || batch < 0 || ssm < 0)
    return set_error(OSSM_ERR_INVALID_ARGUMENT, "dlinoss_backward_f64: negative size");
  if (ssm == 0) return OSSM_OK;
  if (!grad_a || !grad_g || !grad_step)
    return set_error(OSSM_ERR_INVALID_ARGUMENT, "dlinoss_backward_f64: null pointer");
  if (length == 0 || batch == 0) {
    // nothing to scan: zero parameter gradients (the reference's zeros_like)
    double* const outs[3] = {grad_a, grad_g, grad_step};
    for (double* o : outs) {
      hipLaunchKernelGGL(sdl64_zero_kernel, dim3(blocks_for(ssm)), dim3(kBlock64), 0, stream, o,
                         static_cast<long long>(ssm));
      if (int rc = launch_check("sdl64_zero_kernel")) return rc;
    }
    return OSSM_OK;
  }
  if (length > INT_MAX / 2 || batch * ssm > INT_MAX / 2 || length * batch * ssm > (int64_t(1) << 40))
    return set_error(OSSM_ERR_UNSUPPORTED, "dlinoss_backward_f64: size exceeds 32-bit indexing");
  if (!a_diag || !g_diag || !step || !bu || !states || !grad_output || !grad_bu)
    return set_error(OSSM_ERR_INVALID_ARGUMENT, "dlinoss_backward_f64: null pointer");
  const DlParams64 prm{a_diag, g_diag, step, static_cast<int>(ssm)};
  const int64_t nc = batch * ssm;
  Plan64 pl{};
  double* part = nullptr;
  if (int rc = plan64(call, length, nc, false, Dl64<OSSM_DLINOSS_IMEX1>::kBwd, length * nc * 80,
                      [&](int n) { return static_cast<size_t>(n) * nc * 6; }, &pl, &part))
    return rc;
  const int64_t rows = int64_t(pl.n_chunks) * batch;  // of P oscillators' sums each
  if (rows > INT_MAX) return set_error(OSSM_ERR_UNSUPPORTED, "dlinoss_backward_f64: size exceeds 32-bit indexing");
  const unsigned blocks = static_cast<unsigned>((ssm + kSumCols - 1) / kSumCols);
  switch (variant) {
#define OSSM_DL64_BWD(V)                                                                              \
  case V:                                                                                             \
    if (int rc = run_backward64<Dl64<V>>(prm, bu, states, grad_output, grad_bu, NoGrads64{}, part,    \
                                         pl, stream))                                                 \
      return rc;                                                                                      \
    hipLaunchKernelGGL(dl64_param_kernel<V>, dim3(blocks), dim3(kBlock64), 0, stream, prm, part,      \
                       grad_a, grad_g, grad_step, static_cast<int>(rows));                            \
    break;
    OSSM_DL64_BWD(OSSM_DLINOSS_IMEX1)
    OSSM_DL64_BWD(OSSM_DLINOSS_IMEX2)
    OSSM_DL64_BWD(OSSM_DLINOSS_IM)
    OSSM_DL64_BWD(OSSM_DLINOSS_EX)
#undef OSSM_DL64_BWD
  }
  return launch_check("dl64_param_kernel");
}

}  // extern "C"
