// y = x W^T for a handful of rows (one token of each of up to 16 sequences): the projections around the attention of a
// generation step.  Several weight matrices share one launch and every output column goes where its consumer reads it,
// so the step's keys and values are written straight into the cache.
#include "mfma_common.hpp"

namespace segpt {
namespace {

typedef float f32x4c __attribute__((ext_vector_type(4)));

// One workgroup = 16 output columns (rows of a weight matrix) of all rows of x; its eight waves share out the 32-column
// steps of the contraction and add up through LDS in a fixed order.  v_mfma_f32_16x16x32_bf16: A = weight rows (row = lane %
// 16, 8 entries from 8 (lane / 16) on), B = rows of x, C: column = row of x, row = 4 (lane / 16) + r.
//
// Bound by latency, then by HBM: the weights are read once and a wave has all its pieces (up to kBatch steps of 1 KB, K =
// 2048 in one batch) in flight before it waits.  16 columns a workgroup make 122 workgroups of the 1938 columns of an 18 / 6
// head projection with its gate; fewer columns would leave lanes of the matrix instruction idle without more bytes in flight.
// A whole step with its cache (18 / 6 heads of 64; the library's products and an append launch before), us: one sequence of 4096
// keys 102.6 -> 28.9, 16 of 8192 keys 101 -> 49, 16 of 2000 keys at 16 / 16 heads of 128 104 -> 33; more rows than a tile has
// keep the library's products.
constexpr int kWaves = 8, kThreads = 64 * kWaves, kCols = 16, kStep = 32, kBatch = 8;

__global__ __launch_bounds__(kThreads) void linear_rows_kernel(segpt_linear_rows_params p) {
  __shared__ float part[kWaves][kCols][kMaxLinearRows + 1];
  const int tid = threadIdx.x, lane = tid & 63;
  const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
  int tile = blockIdx.x, s = 0;
  while (s + 1 < p.n_segments && tile >= (p.seg[s].n + kCols - 1) / kCols) tile -= (p.seg[s++].n + kCols - 1) / kCols;
  const segpt_linear_segment seg = p.seg[s];
  const int c0 = tile * kCols, r = lane & 15, k0 = 8 * (lane >> 4);
  const uint16_t* w = reinterpret_cast<const uint16_t*>(seg.w) + (int64_t)min(c0 + r, seg.n - 1) * seg.w_stride + k0;
  const uint16_t* x = reinterpret_cast<const uint16_t*>(p.x) + (int64_t)min(r, p.M - 1) * p.x_stride + k0;
  const int steps = p.K / kStep, mine = (steps - wave + kWaves - 1) / kWaves;  // this wave's: wave, wave + 8, ...
  f32x4c acc = {0.f, 0.f, 0.f, 0.f};
  for (int i0 = 0; i0 < mine; i0 += kBatch) {
    u32x4 wf[kBatch], xf[kBatch];
#pragma unroll
    for (int u = 0; u < kBatch; ++u) {
      const int at = (wave + kWaves * min(i0 + u, mine - 1)) * kStep;  // past the end: the last piece once more, unused
      wf[u] = *reinterpret_cast<const u32x4*>(w + at);
      xf[u] = *reinterpret_cast<const u32x4*>(x + at);
    }
#pragma unroll
    for (int u = 0; u < kBatch; ++u)
      if (i0 + u < mine) acc = __builtin_amdgcn_mfma_f32_16x16x32_bf16(as_bf16x8(wf[u]), as_bf16x8(xf[u]), acc, 0, 0, 0);
  }
#pragma unroll
  for (int i = 0; i < 4; ++i) part[wave][4 * (lane >> 4) + i][r] = acc[i];
  __syncthreads();
  const int c = tid % kCols, m = tid / kCols;  // neighbouring threads store neighbouring columns
  if (m >= p.M || c0 + c >= seg.n) return;
  float t[kWaves];
#pragma unroll
  for (int i = 0; i < kWaves; ++i) t[i] = part[i][c][m];
  const float y = ((t[0] + t[1]) + (t[2] + t[3])) + ((t[4] + t[5]) + (t[6] + t[7]));
  const int col = c0 + c, head = col / seg.width;
  reinterpret_cast<uint16_t*>(seg.out)[(int64_t)m * seg.stride_m + (int64_t)head * seg.stride_h + (col - head * seg.width)] =
      (uint16_t)pack_bf16x2(y, y);
}

}  // namespace

int launch_linear_rows(const segpt_linear_rows_params& p, hipStream_t st) {
  int tiles = 0;
  for (int s = 0; s < p.n_segments; ++s) tiles += (p.seg[s].n + kCols - 1) / kCols;
  hipLaunchKernelGGL(linear_rows_kernel, dim3((unsigned)tiles), dim3(kThreads), 0, st, p);
  return (int)hipGetLastError();
}

}  // namespace segpt
