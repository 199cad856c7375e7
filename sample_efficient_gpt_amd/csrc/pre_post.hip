// HBM-bound helper kernels:
//   kv_prep     (bf16 path, forward and backward) the normalised keys Khat and mixed values V' that the MFMA
//               kernels stream, so that their inner loops carry no norm arithmetic.
//   bwd_reduce  (value residual only) sums the per-workgroup (dc1, dc2) partials of the kernel that wrote dV.  The
//               scale-vector gradient is added up by one extra workgroup of the last backward kernel.
#include "common.hpp"

namespace segpt {
namespace {

// bf16 path: Khat = b_j k_j and (with a value residual) V' = c1 v + c2 v_first, one row per 8/16 lanes
template <int D>
__global__ __launch_bounds__(256) void kv_prep_kernel(KArgs a) {
  const segpt_attn_params& p = a.p;
  constexpr int TPR = D / 8;
  constexpr int RPB = 256 / TPR;
  const int tid = threadIdx.x;
  const int part = tid % TPR;
  const int64_t rid = (int64_t)blockIdx.x * RPB + tid / TPR;  // flat (b, g, s)
  const int64_t nrows = (int64_t)p.B * p.Hkv * p.Sk;
  const bool live = rid < nrows;
  const int64_t r = live ? rid : nrows - 1;
  const int s = (int)(r % p.Sk);
  const int g = (int)((r / p.Sk) % p.Hkv);
  const int b = (int)(r / ((int64_t)p.Sk * p.Hkv));
  float k[8];
  Elem<uint16_t>::load(row_ptr<uint16_t>(p.k, b, g, s) + part * 8, k);
  if (p.rope_cos) {
    // split-half pairs (j, j + D/2): the partner element sits TPR/2 lanes away, same slot.  The lane's eight table
    // entries come in as four 16-byte loads (table rows are 16-byte aligned and jp is a multiple of 8 floats) and the
    // two halves share one expression, x' = x c + sign * partner * s, so that no lane-dependent branch splits the loads.
    const int jp = (part % (TPR / 2)) * 8;
    const float* cr = p.rope_cos + (int64_t)(p.rope_k_pos0 + s) * (D / 2) + jp;
    const float* sr = p.rope_sin + (int64_t)(p.rope_k_pos0 + s) * (D / 2) + jp;
    const float4 c0 = *reinterpret_cast<const float4*>(cr), c1 = *reinterpret_cast<const float4*>(cr + 4);
    const float4 s0 = *reinterpret_cast<const float4*>(sr), s1 = *reinterpret_cast<const float4*>(sr + 4);
    const float cv[8] = {c0.x, c0.y, c0.z, c0.w, c1.x, c1.y, c1.z, c1.w};
    const float sv[8] = {s0.x, s0.y, s0.z, s0.w, s1.x, s1.y, s1.z, s1.w};
    const float sign = part < TPR / 2 ? -1.f : 1.f;
#pragma unroll
    for (int e = 0; e < 8; ++e) {
      const float other = __shfl_xor(k[e], TPR / 2, 64);
      k[e] = k[e] * cv[e] + sign * other * sv[e];
    }
  }
  float ss = 0.f;
#pragma unroll
  for (int e = 0; e < 8; ++e) ss += k[e] * k[e];
#pragma unroll
  for (int o = 1; o < TPR; o <<= 1) ss += __shfl_xor(ss, o, 64);
  const float beta = row_normaliser(p, ss, 1.0f / D);
#pragma unroll
  for (int e = 0; e < 8; ++e) k[e] *= beta;
  if (live) Elem<uint16_t>::store(a.khat + r * D + part * 8, k);
  if (a.vmix) {
    const float c1 = p.vr_coef[0], c2 = p.vr_coef[1];
    float v[8], f[8];
    Elem<uint16_t>::load(row_ptr<uint16_t>(p.v, b, g, s) + part * 8, v);
    Elem<uint16_t>::load(row_ptr<uint16_t>(p.v_first, b, g, s) + part * 8, f);
#pragma unroll
    for (int e = 0; e < 8; ++e) v[e] = c1 * v[e] + c2 * f[e];
    if (live) Elem<uint16_t>::store(a.vmix + r * D + part * 8, v);
  }
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
int launch_kv_prep(const KArgs& a, hipStream_t st) {
  const segpt_attn_params& p = a.p;
  const int64_t nrows = (int64_t)p.B * p.Hkv * p.Sk;
  const int rpb = 256 / (p.D / 8);
  dim3 grid((unsigned)((nrows + rpb - 1) / rpb)), block(256);
  if (p.D == 64) hipLaunchKernelGGL(kv_prep_kernel<64>, grid, block, 0, st, a);
  else hipLaunchKernelGGL(kv_prep_kernel<128>, grid, block, 0, st, a);
  return (int)hipGetLastError();
}

int launch_bwd_reduce(const KArgs& a, hipStream_t st) {
  if (!a.p.vr_coef) return 0;  // nothing left to reduce
  hipLaunchKernelGGL(bwd_reduce_kernel, dim3(1), dim3(kReduceThreads), 0, st, a);
  return (int)hipGetLastError();
}

}  // namespace segpt
