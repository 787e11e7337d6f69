// out[m, n] = sum_r a[r, m] b[r, n] for row-major a [R, M], b [R, N] with R much
// larger than M and N: the weight gradients of layers, which sum over every
// (batch, step) row.
//
// Each wave owns a 128 x 64 tile of the output and every (slices * kWaves)-th
// block of 16 rows.  Row-major operands are what the matrix cores want here
// without a transpose: lane l reads 4 columns of a (2 of b) of each of 8 rows,
// lane half l / 32 the rows' half, and column 4 (l % 32) + j is row l % 32 of
// the j-th of the tile's fragments, so a wave reads 512-byte runs straight into
// the fragments' registers and the tile's rows only come out permuted.  Products are
// split into bf16 terms (split_mfma.hpp).  The workgroup's waves add their tiles
// through LDS, and rows_product_sum_kernel adds the slices' tiles in order
// (bitwise repeatable).
//
// Bound: the matrix cores and the splitting together, 48 instructions of 32
// cycles and 264 VALU per 16 rows and tile (0.9 PFLOP/s of bf16 at [131072, 256, 128],
// loads one block ahead; an 8192^3 bf16 product of the library reaches 1.2).  Against
// the library's fp32 GEMM on the same operands, us
// (and its relative error against float64): [51200, 256, 64] 164 -> 24
// (2.5e-6 -> 2.8e-7); [51200, 128, 4] 71 -> 18; [131072, 256, 128] 345 -> 58
// (4e-6 -> 4.3e-7; as 32 batched slices 75, 1.1e-6); [32768, 3072, 768]
// 2388 -> 1340; [1000, 256, 64] 60 -> 14.

#include <hip/hip_runtime.h>

#include <algorithm>
#include <climits>
#include <cstdint>
#include <string>

#include "../../include/ossm_scan.h"
#include "runtime.hpp"
#include "scan_device.hpp"
#include "split_mfma.hpp"

namespace ossm {
namespace {

constexpr int kTm = 128, kTn = 64;  // output tile of a wave
constexpr int kRpWaves = 8;
constexpr int kRpThreads = kRpWaves * kWave;
constexpr int kBlockRows = 16;

struct RowsProduct {
  const float* a;
  const float* b;
  float* part;  // [slices][tiles][kTm][kTn]
  long long R, lda, ldb;
  int M, N, tiles_m, tiles_n, slices;
};

// W columns of a row from the lane's offsets, V at a time (V = W: one aligned vector
// load; 2: pairs, for even widths that are no multiple of 4).
template <int V, int W>
__device__ __forceinline__ void load_cols(const float* __restrict__ row, const unsigned (&off)[W],
                                          float (&v)[W]) {
  if constexpr (V == 1) {
#pragma unroll
    for (int j = 0; j < W; ++j) v[j] = row[off[j]];
  } else {
    typedef float X __attribute__((ext_vector_type(V)));
#pragma unroll
    for (int q = 0; q < W; q += V) {
      const X x = *reinterpret_cast<const X*>(row + off[q]);
#pragma unroll
      for (int j = 0; j < V; ++j) v[q + j] = x[j];
    }
  }
}

// The lane's column j of W from c0, clamped in range V columns at a time.
template <int V>
__device__ __forceinline__ unsigned clamp_col(int c0, int j, int n) {
  return static_cast<unsigned>(min(c0 + j / V * V, n - V) + j % V);
}

// A wave's tile in fp32, for sums that left the range of the split products
// (split_mfma.hpp).
__device__ __forceinline__ void exact_tile(const RowsProduct& g, int slice, int m0, int n0, floatx16 (&acc)[4][2]) {
  int lane = threadIdx.x & (kWave - 1);
  asm volatile("" : "+v"(lane));  // keeps this path's values out of the main loop's registers
  const int half = lane >> 5, l32 = lane & 31;
#pragma unroll
  for (int i = 0; i < 4; ++i)
#pragma unroll
    for (int j = 0; j < 2; ++j)
#pragma unroll
      for (int r = 0; r < 16; ++r) acc[i][j][r] = 0.f;
  const long long n_blocks = (g.R + kBlockRows - 1) / kBlockRows;
  for (long long blk = static_cast<long long>(slice) * kRpWaves + wave_id(); blk < n_blocks;
       blk += static_cast<long long>(g.slices) * kRpWaves) {
#pragma unroll 1
    for (int i = 0; i < 8; ++i) {
      const long long row = blk * kBlockRows + 8 * half + i;
      const bool in = row < g.R;
      const float* pa = g.a + min(row, g.R - 1) * g.lda;
      const float* pb = g.b + min(row, g.R - 1) * g.ldb;
      float va[4], vb[2];
#pragma unroll
      for (int j = 0; j < 4; ++j) va[j] = in ? pa[clamp_col<1>(m0 + 4 * l32, j, g.M)] : 0.f;
#pragma unroll
      for (int j = 0; j < 2; ++j) vb[j] = in ? pb[clamp_col<1>(n0 + 2 * l32, j, g.N)] : 0.f;
#pragma unroll
      for (int j = 0; j < 4; ++j)
#pragma unroll
        for (int k = 0; k < 2; ++k) acc[j][k] = mfma32(va[j], vb[k], acc[j][k]);
    }
  }
}

// VA, VB: columns of a and b loaded at once.
template <int VA, int VB>
__global__ __launch_bounds__(kRpThreads, 1) __attribute__((amdgpu_waves_per_eu(2, 2)))
void rows_product_kernel(RowsProduct g) {
  extern __shared__ __align__(16) float s_tile[];  // [kRpWaves / 2][kTm * kTn]
  const int lane = threadIdx.x & (kWave - 1), w = wave_id();
  const int half = lane >> 5, l32 = lane & 31;
  // consecutive ids share an XCD (dispatch is round-robin over the 8 of them),
  // and the tiles of one slice are consecutive: they read the same rows
  const int total = static_cast<int>(gridDim.x);
  const int per = total / 8;
  const int bid = static_cast<int>(blockIdx.x);
  const int id = bid < per * 8 ? (bid % 8) * per + bid / 8 : bid;
  const int tiles = g.tiles_m * g.tiles_n;
  const int slice = id / tiles, tile = id - slice * tiles;
  const int m0 = (tile / g.tiles_n) * kTm, n0 = (tile % g.tiles_n) * kTn;
  // lane offsets from the block's first row; columns out of range read clamped
  // ones, which only reach outputs that are not stored
  unsigned oa[4], ob[2];
#pragma unroll
  for (int j = 0; j < 4; ++j)
    oa[j] = static_cast<unsigned>(8 * half * g.lda) + clamp_col<VA>(m0 + 4 * l32, j, g.M);
#pragma unroll
  for (int j = 0; j < 2; ++j)
    ob[j] = static_cast<unsigned>(8 * half * g.ldb) + clamp_col<VB>(n0 + 2 * l32, j, g.N);

  floatx16 acc[4][2];
#pragma unroll
  for (int i = 0; i < 4; ++i)
#pragma unroll
    for (int j = 0; j < 2; ++j)
#pragma unroll
      for (int r = 0; r < 16; ++r) acc[i][j][r] = 0.f;

  const long long n_blocks = (g.R + kBlockRows - 1) / kBlockRows;
  const long long stride = static_cast<long long>(g.slices) * kRpWaves;
  long long blk = static_cast<long long>(slice) * kRpWaves + w;
  float ra[8][4], rb[8][2];
  // a short last block is loaded from R - 16 (its first rows belong to the block
  // before and are zeroed), so every row is in range and its address uniform
  auto load = [&](long long k) {
    const long long r0 = min(k * kBlockRows, g.R - kBlockRows);
#pragma unroll
    for (int i = 0; i < 8; ++i) {
      load_cols<VA, 4>(g.a + (r0 + i) * g.lda, oa, ra[i]);
      load_cols<VB, 2>(g.b + (r0 + i) * g.ldb, ob, rb[i]);
    }
  };
  if (blk < n_blocks) load(blk);
  for (; blk < n_blocks; blk += stride) {
    if (blk == n_blocks - 1) {
      const int done = static_cast<int>(n_blocks * kBlockRows - g.R);
#pragma unroll
      for (int i = 0; i < 8; ++i) {
        if (8 * half + i < done) {
#pragma unroll
          for (int j = 0; j < 4; ++j) ra[i][j] = 0.f;
          rb[i][0] = rb[i][1] = 0.f;
        }
      }
    }
    SplitFrag fb[2], fa[4];
#pragma unroll
    for (int j = 0; j < 2; ++j) {
      float x[8];
#pragma unroll
      for (int i = 0; i < 8; ++i) x[i] = rb[i][j];
      fb[j] = split8(x);
    }
#pragma unroll
    for (int j = 0; j < 4; ++j) {
      float x[8];
#pragma unroll
      for (int i = 0; i < 8; ++i) x[i] = ra[i][j];
      fa[j] = split8(x);
    }
    load(min(blk + stride, n_blocks - 1));  // in flight under the products
    __builtin_amdgcn_sched_barrier(0);
    // term by term over the eight products: consecutive instructions are independent
    const auto term = [&](auto ta, auto tb) {
#pragma unroll
      for (int i = 0; i < 4; ++i)
#pragma unroll
        for (int j = 0; j < 2; ++j) acc[i][j] = mfma_bf16(ta(fa[i]), tb(fb[j]), acc[i][j]);
    };
    const auto t0 = [](const SplitFrag& f) { return f.t0; };
    const auto t1 = [](const SplitFrag& f) { return f.t1; };
    const auto t2 = [](const SplitFrag& f) { return f.t2; };
    term(t2, t0);
    term(t1, t1);
    term(t0, t2);
    term(t1, t0);
    term(t0, t1);
    term(t0, t0);
  }

  if (any_nonfinite(acc[0]) || any_nonfinite(acc[1]) || any_nonfinite(acc[2]) || any_nonfinite(acc[3]))
    exact_tile(g, slice, m0, n0, acc);

  // The workgroup's tile.  Waves 4-7 hand theirs to waves 0-3 through LDS, then
  // all waves add those four, 16 elements per thread (three halving rounds
  // of single-word accesses took 12 of 24 us at [51200, 256, 64]).
  // Element order: 16-byte runs of four accumulator registers, lanes adjacent.
  constexpr int kTile = kTm * kTn;
  typedef float f32x4 __attribute__((ext_vector_type(4)));
  auto* s4 = reinterpret_cast<f32x4*>(s_tile);
  const auto put = [&](f32x4* dst) {
#pragma unroll
    for (int i = 0; i < 4; ++i)
#pragma unroll
      for (int j = 0; j < 2; ++j)
#pragma unroll
        for (int q = 0; q < 4; ++q) {
          const floatx16& v = acc[i][j];
          dst[((i * 2 + j) * 4 + q) * kWave + lane] = f32x4{v[4 * q], v[4 * q + 1], v[4 * q + 2], v[4 * q + 3]};
        }
  };
  constexpr int kHalf = kRpWaves / 2;
  if (w >= kHalf) put(s4 + (w - kHalf) * (kTile / 4));
  __syncthreads();
  if (w < kHalf) {
    f32x4* mine = s4 + w * (kTile / 4);
#pragma unroll
    for (int i = 0; i < 4; ++i)
#pragma unroll
      for (int j = 0; j < 2; ++j)
#pragma unroll
        for (int q = 0; q < 4; ++q) {
          const f32x4 o = mine[((i * 2 + j) * 4 + q) * kWave + lane];
#pragma unroll
          for (int x = 0; x < 4; ++x) acc[i][j][4 * q + x] += o[x];
        }
    put(mine);  // its own slot: no other wave reads it before the barrier
  }
  __syncthreads();
  auto* dst = reinterpret_cast<f32x4*>(g.part + (static_cast<size_t>(slice) * tiles + tile) * kTile);
#pragma unroll
  for (int k = 0; k < kTile / 4 / kRpThreads; ++k) {
    const int e = k * kRpThreads + static_cast<int>(threadIdx.x);
    f32x4 v = s4[e];
#pragma unroll
    for (int u = 1; u < kHalf; ++u) v += s4[u * (kTile / 4) + e];
    dst[e] = v;
  }
}

// out(m, n) = the slices' sums, at out[(m / 2) s_pair + (m % 2) s_odd + n s_n]:
// plain row-major is (2 ld, ld, 1), and pairs of rows may interleave.
struct RowsOut {
  float* out;
  long long s_pair, s_odd, s_n;
};

constexpr int kSumBlock = 256, kSumLanes = 4;  // 64 outputs per workgroup, 4 lanes of slices each

__global__ __launch_bounds__(kSumBlock) void rows_product_sum_kernel(const float* __restrict__ part, int M,
                                                                     int N, int tiles_n, int tiles, int slices,
                                                                     RowsOut o) {
  __shared__ float s_p[kSumLanes][kWave];
  const int e = static_cast<int>(blockIdx.x) * kWave + static_cast<int>(threadIdx.x & (kWave - 1));
  const int sl = static_cast<int>(threadIdx.x) / kWave;
  float s = 0.f;
  const size_t stride = static_cast<size_t>(tiles) * (kTm * kTn);
#pragma unroll 8
  for (int k = sl; k < slices; k += kSumLanes) s += part[k * stride + e];
  s_p[sl][threadIdx.x & (kWave - 1)] = s;
  __syncthreads();
  if (sl != 0) return;
#pragma unroll
  for (int v = 1; v < kSumLanes; ++v) s += s_p[v][threadIdx.x];
  // element e of the tiles: fragment (i, j), accumulator register r, lane l
  const int tile = e / (kTm * kTn), q = e % (kTm * kTn);
  const int r = (q & 3) + 4 * ((q >> 8) & 3), l = (q >> 2) & (kWave - 1), j = (q >> 10) & 1, i = q >> 11;
  const int row = 8 * (r >> 2) + 4 * (l >> 5) + (r & 3);  // of the 32 x 32 fragment product
  const int m = (tile / tiles_n) * kTm + 4 * row + i, n = (tile % tiles_n) * kTn + 2 * (l & 31) + j;
  if (m < M && n < N) o.out[(m >> 1) * o.s_pair + (m & 1) * o.s_odd + n * o.s_n] = s;
}

bool aligned_to(const void* p, size_t n) { return (reinterpret_cast<uintptr_t>(p) & (n - 1)) == 0; }

}  // namespace
}  // namespace ossm

using namespace ossm;

extern "C" {

int ossm_rows_product(const float* a, int64_t ld_a, const float* b, int64_t ld_b, float* out,
                      int64_t out_pair_stride, int64_t out_odd_stride, int64_t out_col_stride, int64_t rows,
                      int64_t m, int64_t n, ossm_stream_t stream_v) {
  clear_error();
  const char* what = "rows_product";
  hipStream_t stream = static_cast<hipStream_t>(stream_v);
  StreamCall call(stream);
  if (call.status()) return call.status();
  if (rows < 0 || m < 0 || n < 0 || ld_a < m || ld_b < n)
    return set_error(OSSM_ERR_INVALID_ARGUMENT, std::string(what) + ": bad size or row stride");
  if (m == 0 || n == 0) return OSSM_OK;
  if (rows < kBlockRows || ld_a > (1 << 26) || ld_b > (1 << 26))
    return set_error(OSSM_ERR_UNSUPPORTED, std::string(what) + ": at least 16 rows, strides up to 2^26");
  if (!a || !b || !out) return set_error(OSSM_ERR_INVALID_ARGUMENT, std::string(what) + ": null pointer");
  const int64_t tm = (m + kTm - 1) / kTm, tn = (n + kTn - 1) / kTn, tiles = tm * tn;
  // one workgroup per CU, each wave with at least two blocks of
  // rows (1, 2, 4: 11.1, 12.6, 18.6 us at [8192, 128, 64]; 20.9, 19.8, 20.2 at
  // [51200, 64, 128]: the partial tiles grow with the slices)
  const int64_t blocks = (rows + kBlockRows - 1) / kBlockRows;
  const int64_t cus = std::max(1, device_cu_count(call.device()));
  const int64_t slices = std::max<int64_t>(1, std::min(cus / tiles, blocks / (2 * kRpWaves)));
  const int64_t elems = tiles * kTm * kTn;
  if (tiles * slices > INT_MAX || elems > INT_MAX)
    return set_error(OSSM_ERR_UNSUPPORTED, std::string(what) + ": problem too large for one launch grid");
  void* ws = nullptr;
  if (int rc = acquire_workspace(call, static_cast<size_t>(slices * elems) * sizeof(float), &ws)) return rc;
  const RowsProduct g{a, b, static_cast<float*>(ws), rows, ld_a, ld_b, static_cast<int>(m),
                      static_cast<int>(n), static_cast<int>(tm), static_cast<int>(tn),
                      static_cast<int>(slices)};
  const int va = m % 4 == 0 && ld_a % 4 == 0 && aligned_to(a, 16)  ? 4
                 : m % 2 == 0 && ld_a % 2 == 0 && aligned_to(a, 8) ? 2
                                                                   : 1;
  const bool vb = n % 2 == 0 && ld_b % 2 == 0 && aligned_to(b, 8);
  auto kern = vb ? (va == 4 ? rows_product_kernel<4, 2> : va == 2 ? rows_product_kernel<2, 2> : rows_product_kernel<1, 2>)
                 : (va == 4 ? rows_product_kernel<4, 1> : va == 2 ? rows_product_kernel<2, 1> : rows_product_kernel<1, 1>);
  constexpr int lds = kRpWaves / 2 * kTm * kTn * static_cast<int>(sizeof(float));
  if (int rc = hip_check(hipFuncSetAttribute(reinterpret_cast<const void*>(kern),
                                             hipFuncAttributeMaxDynamicSharedMemorySize, lds),
                         "hipFuncSetAttribute"))
    return rc;
  hipLaunchKernelGGL(kern, dim3(static_cast<unsigned>(tiles * slices)), dim3(kRpThreads), lds, stream, g);
  if (int rc = launch_check("rows_product_kernel")) return rc;
  hipLaunchKernelGGL(rows_product_sum_kernel, dim3(static_cast<unsigned>(elems / kWave)), dim3(kSumBlock), 0,
                     stream, static_cast<const float*>(ws), g.M, g.N, g.tiles_n, static_cast<int>(tiles),
                     g.slices, RowsOut{out, out_pair_stride, out_odd_stride, out_col_stride});
  return launch_check("rows_product_sum_kernel");
}

}  // extern "C"
