// HBM-bound helper kernels:
//   kv_prep     (bf16 path, forward and backward) the normalised keys Khat and mixed values V' that the MFMA
//               kernels stream, so that their inner loops carry no norm arithmetic.
//   bwd_reduce  (value residual only) sums the per-workgroup (dc1, dc2) partials of the kernel that wrote dV.  The
//               scale-vector gradient is added up by one extra workgroup of the last backward kernel.
#include "common.hpp"

namespace segpt {
namespace {

// bf16 path: Khat = b_j k_j and (with a value residual) V' = c1 v + c2 v_first.  Bound by HBM (a row is read and written
// once): 8 / 16 lanes per row, two rows per thread so that a wave has twice the bytes in flight and 8 x 2048 tokens of 6 kv heads
// are one resident round; (batch, kv head) comes from the grid instead of 64-bit divisions per thread, and what the call
// does not have (ROPE: tables, MIX: a value residual) is no branch between the loads.  8 x 2048 x 6 rows of 64: 6.4 -> 5.1 us,
// with tables and residual 12.5 -> 10.9; 4 x 4096 x 4 rows of 128: 7.8 -> 5.9; 1 x 8192 x 6 with tables: 4.8 -> 4.4; 1 x 512 x 6: 2.6 (the launch).
constexpr int kPrepRows = 2;  // rows per thread
template <int D, bool ROPE, bool MIX>
__global__ __launch_bounds__(256) void kv_prep_kernel(KArgs a) {
  const segpt_attn_params& p = a.p;
  constexpr int TPR = D / 8;
  constexpr int RPB = 256 / TPR;
  const int tid = threadIdx.x;
  const int part = tid % TPR;
  const int g = blockIdx.y, b = blockIdx.z;
  int s[kPrepRows];
  bool live[kPrepRows];
  float k[kPrepRows][8], v[kPrepRows][8], f[kPrepRows][8];
#pragma unroll
  for (int u = 0; u < kPrepRows; ++u) {
    s[u] = (int)blockIdx.x * (RPB * kPrepRows) + u * RPB + tid / TPR;
    live[u] = s[u] < p.Sk;
    s[u] = min(s[u], p.Sk - 1);
    Elem<uint16_t>::load(row_ptr<uint16_t>(p.k, b, g, s[u]) + part * 8, k[u]);
    if (MIX) {
      Elem<uint16_t>::load(row_ptr<uint16_t>(p.v, b, g, s[u]) + part * 8, v[u]);
      Elem<uint16_t>::load(row_ptr<uint16_t>(p.v_first, b, g, s[u]) + part * 8, f[u]);
    }
  }
  float cv[kPrepRows][8], sv[kPrepRows][8];
  if (ROPE) {
    // split-half pairs (j, j + D/2): the partner element sits TPR/2 lanes away, same slot.  The lane's eight table
    // entries come in as four 16-byte loads (table rows are 16-byte aligned and jp is a multiple of 8 floats) and the
    // two halves share one expression, x' = x c + sign * partner * s, so that no lane-dependent branch splits the loads.
    const int jp = (part % (TPR / 2)) * 8;
#pragma unroll
    for (int u = 0; u < kPrepRows; ++u) {
      const float* cr = p.rope_cos + (int64_t)(p.rope_k_pos0 + s[u]) * (D / 2) + jp;
      const float* sr = p.rope_sin + (int64_t)(p.rope_k_pos0 + s[u]) * (D / 2) + jp;
#pragma unroll
      for (int e = 0; e < 8; e += 4) {
        const float4 c4 = *reinterpret_cast<const float4*>(cr + e), s4 = *reinterpret_cast<const float4*>(sr + e);
        cv[u][e] = c4.x; cv[u][e + 1] = c4.y; cv[u][e + 2] = c4.z; cv[u][e + 3] = c4.w;
        sv[u][e] = s4.x; sv[u][e + 1] = s4.y; sv[u][e + 2] = s4.z; sv[u][e + 3] = s4.w;
      }
    }
  }
  float c1 = 1.f, c2 = 0.f;
  if (MIX) { c1 = p.vr_coef[0]; c2 = p.vr_coef[1]; }
#pragma unroll
  for (int u = 0; u < kPrepRows; ++u) {
    if (ROPE) {
      const float sign = part < TPR / 2 ? -1.f : 1.f;
#pragma unroll
      for (int e = 0; e < 8; ++e) {
        const float other = __shfl_xor(k[u][e], TPR / 2, 64);
        k[u][e] = k[u][e] * cv[u][e] + sign * other * sv[u][e];
      }
    }
    float ss = 0.f;
#pragma unroll
    for (int e = 0; e < 8; ++e) ss += k[u][e] * k[u][e];
#pragma unroll
    for (int o = 1; o < TPR; o <<= 1) ss += __shfl_xor(ss, o, 64);
    const float beta = row_normaliser(p, ss, 1.0f / D);
    const int64_t at = (((int64_t)b * p.Hkv + g) * p.Sk + s[u]) * D + part * 8;
#pragma unroll
    for (int e = 0; e < 8; ++e) k[u][e] *= beta;
    if (live[u]) Elem<uint16_t>::store(a.khat + at, k[u]);
    if (MIX) {
#pragma unroll
      for (int e = 0; e < 8; ++e) v[u][e] = c1 * v[u][e] + c2 * f[u][e];
      if (live[u]) Elem<uint16_t>::store(a.vmix + at, v[u]);
    }
  }
}

// One step's rows of k and v behind the rows of a cache.  A generation step appends a kilobyte: what counts is that both
// tensors are ONE launch (two copies of 2.3 us each and their dispatch before, 2.3 us now); a prompt is bound by HBM.
constexpr int kAppendThreads = 64;
__global__ __launch_bounds__(kAppendThreads) void kv_append_kernel(KvAppendArgs a) {
  const int i = blockIdx.x * kAppendThreads + threadIdx.x;
  if (i >= a.S * a.chunks) return;
  const int s = i / a.chunks, c = i - s * a.chunks;
  const int t = blockIdx.y & 1, g = blockIdx.y >> 1, b = blockIdx.z;
  const char* src = a.src[t] + b * a.src_b[t] + g * a.src_h[t] + s * a.src_s[t] + 16 * c;
  char* dst = a.dst[t] + b * a.dst_b[t] + g * a.dst_h[t] + s * a.dst_s[t] + 16 * c;
  *reinterpret_cast<uint4*>(dst) = *reinterpret_cast<const uint4*>(src);
}

constexpr int kReduceThreads = 1024;

__global__ __launch_bounds__(kReduceThreads) void bwd_reduce_kernel(KArgs a) {
  const segpt_attn_params& p = a.p;
  __shared__ float red[kReduceThreads / 64 * 2];
  const int tid = threadIdx.x;
  float s1 = 0.f, s2 = 0.f;
  for (int b2 = tid; b2 < a.n_dkdv_blocks; b2 += kReduceThreads) {
    s1 += a.dcoef_part[(int64_t)b2 * 2];
    s2 += a.dcoef_part[(int64_t)b2 * 2 + 1];
  }
#pragma unroll
  for (int o = 1; o < 64; o <<= 1) { s1 += __shfl_xor(s1, o, 64); s2 += __shfl_xor(s2, o, 64); }
  if ((tid & 63) == 0) { red[(tid >> 6) * 2] = s1; red[(tid >> 6) * 2 + 1] = s2; }
  __syncthreads();
  if (tid < 2) {
    float t = 0.f;
    for (int w = 0; w < kReduceThreads / 64; ++w) t += red[w * 2 + tid];
    p.dvr_coef[tid] = t;
  }
}

}  // namespace

// bf16: the per-key-row pre-pass shared by forward and backward (the per-query-row quantities of the backward,
// delta / Qhat / gate terms, come from the dQ kernel's prologue)
template <int D>
static void launch_kv_prep_t(const KArgs& a, hipStream_t st) {
  const segpt_attn_params& p = a.p;
  constexpr int rows = 256 / (D / 8) * kPrepRows;
  const dim3 grid((unsigned)((p.Sk + rows - 1) / rows), (unsigned)p.Hkv, (unsigned)p.B), block(256);
  if (p.rope_cos) {
    if (a.vmix) hipLaunchKernelGGL((kv_prep_kernel<D, true, true>), grid, block, 0, st, a);
    else hipLaunchKernelGGL((kv_prep_kernel<D, true, false>), grid, block, 0, st, a);
  } else {
    if (a.vmix) hipLaunchKernelGGL((kv_prep_kernel<D, false, true>), grid, block, 0, st, a);
    else hipLaunchKernelGGL((kv_prep_kernel<D, false, false>), grid, block, 0, st, a);
  }
}
int launch_kv_prep(const KArgs& a, hipStream_t st) {
  if (a.p.D == 64) launch_kv_prep_t<64>(a, st);
  else launch_kv_prep_t<128>(a, st);
  return (int)hipGetLastError();
}

int launch_kv_append(const KvAppendArgs& a, hipStream_t st) {
  const dim3 grid((unsigned)((a.S * a.chunks + kAppendThreads - 1) / kAppendThreads), (unsigned)(2 * a.Hkv), (unsigned)a.B);
  hipLaunchKernelGGL(kv_append_kernel, grid, dim3(kAppendThreads), 0, st, a);
  return (int)hipGetLastError();
}

int launch_bwd_reduce(const KArgs& a, hipStream_t st) {
  if (!a.p.vr_coef) return 0;  // nothing left to reduce
  hipLaunchKernelGGL(bwd_reduce_kernel, dim3(1), dim3(kReduceThreads), 0, st, a);
  return (int)hipGetLastError();
}

}  // namespace segpt
