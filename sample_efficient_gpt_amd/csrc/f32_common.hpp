// Shared by the fp32 kernels: f32_path.hip (fp32 matrix instruction) and f32_split.hip (three-way bf16 splits).
#pragma once

#include "common.hpp"
#include "work_order.hpp"

namespace segpt {

int f32_dq_grid(const segpt_attn_params& p);
int f32_dkdv_splits(const segpt_attn_params& p);

namespace {

typedef float f32x16 __attribute__((ext_vector_type(16)));
typedef float f32x4v __attribute__((ext_vector_type(4)));

constexpr int kRows = 32;      // stationary rows of a workgroup = rows of a streamed tile
constexpr int kWaves = 4;
constexpr int kThreads = 64 * kWaves;
constexpr int kFinishFloats = 4 * kThreads;  // elements of dK one workgroup of the finish kernel owns

template <int D>
struct T32 {
  static constexpr int kLPR = D / 4;            // lanes (16 bytes each) per row
  static constexpr int kRPP = 64 / kLPR;        // rows one wave-wide access covers
  static constexpr int kPasses = kRows / kRPP;  // accesses per tile
  static constexpr int kRS = D + 4;             // row stride in LDS (floats): 16 rows x 16 bytes of an rm read hit 64 banks
  static constexpr int kTile = kRows * kRS;     // floats
  static constexpr int kMB = D / 32;
  static constexpr int kC = D / 8;
  static constexpr int kOcc = D == 128 ? 1 : 2; // workgroups per CU: what two tiles per wave leave of the 160 KB LDS
};

__device__ __forceinline__ f32x16 mfma(float a, float b, f32x16 c) {
  return __builtin_amdgcn_mfma_f32_32x32x2f32(a, b, c, 0, 0, 0);
}
__device__ __forceinline__ f32x16 zero16() {
  f32x16 v;
#pragma unroll
  for (int r = 0; r < 16; ++r) v[r] = 0.f;
  return v;
}
// A dot product over the columns runs as N independent sums, as many as the kernel has registers for: one sum of all D
// products is D roundings deep, and its error grew with D.  Norm-wise distance to float64 of y with one sum, with N: head_dim
// 64, 165 tokens 2.2e-7, 1.6e-7; 128, 212 tokens 2.9e-7, 1.7e-7 (plain FMA loops, four sums a row: 2.0e-7 and 2.1e-7).
// Time: the same (forward 2 x 4 heads, 256 tokens 10.9 -> 11.1 us, step of 2 x 8 heads, 1000 tokens 141.8 -> 142.2).
template <int N>
__device__ __forceinline__ f32x16 add_chains(f32x16 (&s)[N]) {
#pragma unroll
  for (int n = N / 2; n > 0; n /= 2)
#pragma unroll
    for (int i = 0; i < n; ++i)
#pragma unroll
      for (int r = 0; r < 16; ++r) s[i][r] += s[i + n][r];
  return s[0];
}
// probability of a score that carries log2 e, from the row's natural lse: one rounding, of the difference (lse * log2 e
// rounded first is off by half a unit at |lse|, for every key of the row alike)
__device__ __forceinline__ float prob(float s, float lse) { return __builtin_amdgcn_exp2f(fmaf(lse, -kLog2e, s)); }
__device__ __forceinline__ int crow(int r, int hh) { return 8 * (r >> 2) + 4 * hh + (r & 3); }

// LDS regions here are private to a wave: program order is enough, the compiler only has to keep it
__device__ __forceinline__ void wave_sync() {
  __builtin_amdgcn_fence(__ATOMIC_ACQ_REL, "wavefront");
  __builtin_amdgcn_wave_barrier();
}

template <int CTRL>
__device__ __forceinline__ float dpp_add(float x) {
  return x + __int_as_float(__builtin_amdgcn_update_dpp(0, __float_as_int(x), CTRL, 0xf, 0xf, true));
}
__device__ __forceinline__ float half_sum(float x) {
  auto r = __builtin_amdgcn_permlane32_swap(__float_as_uint(x), __float_as_uint(x), false, false);
  return __uint_as_float(r[0]) + __uint_as_float(r[1]);
}
__device__ __forceinline__ float half_max(float x) {
  auto r = __builtin_amdgcn_permlane32_swap(__float_as_uint(x), __float_as_uint(x), false, false);
  return fmaxf(__uint_as_float(r[0]), __uint_as_float(r[1]));
}
// sum over the LPR (8, 16 or 32) consecutive lanes that hold a row
template <int LPR>
__device__ __forceinline__ float row_sum(float x) {
  x = dpp_add<0xB1>(x);   // lane ^ 1
  x = dpp_add<0x4E>(x);   // lane ^ 2
  x = dpp_add<0x141>(x);  // mirrored within 8 lanes
  if (LPR >= 16) x = dpp_add<0x140>(x);  // mirrored within 16
  if (LPR >= 32) {
    auto r = __builtin_amdgcn_permlane16_swap(__float_as_uint(x), __float_as_uint(x), false, false);
    x = __uint_as_float(r[0]) + __uint_as_float(r[1]);
  }
  return x;
}

template <int D>
__device__ __forceinline__ float gprod(const segpt_attn_params& p, int d) {
  float gq = p.gq_numel == 1 ? p.g_q[0] : p.g_q[d];
  float gk = p.gk_numel == 0 ? 1.0f : (p.gk_numel == 1 ? p.g_k[0] : p.g_k[d]);
  return gq * gk;
}

// ---- row-split layout: a row is spread over LPR consecutive lanes, lane `part` of it holds elements 4 part .. + 3

// Split-half rotary embedding (rope.py:50-55): the partner element d +- D/2 sits LPR/2 lanes away, same slot.  `pos` is
// the row's table row; every lane of the wave must get here (the lanes shuffle).  INVERSE applies the transpose.
template <int D, bool INVERSE>
__device__ __forceinline__ f32x4v rope_row(const segpt_attn_params& p, f32x4v x, int pos, int part) {
  constexpr int HL = T32<D>::kLPR / 2;
  const int jp = 4 * (part % HL);
  const f32x4v c = *reinterpret_cast<const f32x4v*>(p.rope_cos + (int64_t)pos * (D / 2) + jp);
  const f32x4v s = *reinterpret_cast<const f32x4v*>(p.rope_sin + (int64_t)pos * (D / 2) + jp);
  const float sign = (part < HL) != INVERSE ? -1.f : 1.f;
  f32x4v y;
#pragma unroll
  for (int e = 0; e < 4; ++e) y[e] = x[e] * c[e] + sign * __shfl_xor(x[e], HL, 64) * s[e];
  return y;
}

// rows row0 .. row0+31 of a [n, D] view as the wave's registers; rows past the end re-read the last one
template <int D>
__device__ __forceinline__ void load_tile(f32x4v (&x)[T32<D>::kPasses], const float* base, int64_t stride_s, int row0, int n, int lane) {
  using T = T32<D>;
  const float* src = base + (int64_t)row0 * stride_s + 4 * (lane % T::kLPR);
  const int last = n - 1 - row0;
#pragma unroll
  for (int ps = 0; ps < T::kPasses; ++ps)
    x[ps] = *reinterpret_cast<const f32x4v*>(src + (int64_t)min(ps * T::kRPP + lane / T::kLPR, last) * stride_s);
}

// 1/sqrt(mean x^2 + eps) of a row from its sum of squares: v_rsq_f32 (1 ulp) and one Newton step, six instructions for
// the divide and square root sequences' forty; exactly 1 for plain attention (`norm` is wave-uniform).  A sum of squares that
// overflowed has y = 0, and so has the result: the median gives the step's NaN a value.  x must be normal
// (v_rsq_f32 flushes others): see TINY_EPS.
__device__ __forceinline__ float inv_rms(float ss, float inv_d, float eps, bool norm) {
  const float x = ss * inv_d + eps;
  const float y = __builtin_amdgcn_rsqf(x);
  return norm ? fmaf(0.5f * y, __builtin_amdgcn_fmed3f(fmaf(-x * y, y, 1.0f), -1.0f, 1.0f), y) : 1.0f;
}
// TINY_EPS: eps is no normal number, so a row's mean square on top of it need not be one either; the kernels then take the
// epilogues' form.  A template parameter: as a branch in the tile loop it cost 3 %.
inline bool tiny_eps(const segpt_attn_params& p) {
  constexpr float kSmallestNormal = 1.17549435e-38f;
  return !(p.flags & SEGPT_FLAG_NO_NORM) && !(p.eps >= kSmallestNormal);
}

// normalise (and rotate) the rows of a tile and put them into LDS: x * 1/rms(x) * scale.  All rows' sums are formed
// side by side, and the one branch (rotary tables or not) stands outside the row loop.  KEEP: they stay in the registers too.
template <int D, bool TINY_EPS, bool KEEP = false>
__device__ __forceinline__ void stage_norm(const segpt_attn_params& p, f32x4v (&x)[T32<D>::kPasses], f32x4v scale, int pos0, int last,
                                           float* tile, int lane) {
  using T = T32<D>;
  const int part = lane % T::kLPR, lr = lane / T::kLPR;
  if (p.rope_cos) {
#pragma unroll
    for (int ps = 0; ps < T::kPasses; ++ps) x[ps] = rope_row<D, false>(p, x[ps], pos0 + min(ps * T::kRPP + lr, last), part);
  }
  const bool norm = !(p.flags & SEGPT_FLAG_NO_NORM);
  float inv[T::kPasses];
#pragma unroll
  for (int ps = 0; ps < T::kPasses; ++ps)
    inv[ps] = row_sum<T::kLPR>((x[ps][0] * x[ps][0] + x[ps][1] * x[ps][1]) + (x[ps][2] * x[ps][2] + x[ps][3] * x[ps][3]));
#pragma unroll
  for (int ps = 0; ps < T::kPasses; ++ps) {
    const float n = TINY_EPS ? row_normaliser(p, inv[ps], 1.0f / D) : inv_rms(inv[ps], 1.0f / D, p.eps, norm);
    const f32x4v y = x[ps] * (n * scale);
    if (KEEP) x[ps] = y;
    *reinterpret_cast<f32x4v*>(tile + (ps * T::kRPP + lr) * T::kRS + 4 * part) = y;
  }
}
template <int D>
__device__ __forceinline__ void stage_plain(const f32x4v (&x)[T32<D>::kPasses], float* tile, int lane) {
  using T = T32<D>;
#pragma unroll
  for (int ps = 0; ps < T::kPasses; ++ps)
    *reinterpret_cast<f32x4v*>(tile + (ps * T::kRPP + lane / T::kLPR) * T::kRS + 4 * (lane % T::kLPR)) = x[ps];
}

// V' = c1 v + c2 v_first of a tile
template <int D>
__device__ __forceinline__ void load_vmix(const segpt_attn_params& p, f32x4v (&x)[T32<D>::kPasses], int b, int g, int row0, float c1, float c2, int lane) {
  load_tile<D>(x, row_ptr<float>(p.v, b, g, 0), p.v.stride_s, row0, p.Sk, lane);
  if (p.v_first.ptr) {
    f32x4v f[T32<D>::kPasses];
    load_tile<D>(f, row_ptr<float>(p.v_first, b, g, 0), p.v_first.stride_s, row0, p.Sk, lane);
#pragma unroll
    for (int ps = 0; ps < T32<D>::kPasses; ++ps)
#pragma unroll
      for (int e = 0; e < 4; ++e) x[ps][e] = c1 * x[ps][e] + c2 * f[ps][e];
  }
}

template <int D>
__device__ __forceinline__ f32x4v frag_rm(const float* tile, int c, int lane) {
  return *reinterpret_cast<const f32x4v*>(tile + (lane & 31) * T32<D>::kRS + 8 * c + 4 * (lane >> 5));
}
template <int D>
struct FragTr {
  float v[T32<D>::kMB];
};
template <int D>
__device__ __forceinline__ FragTr<D> frag_tr(const float* tile, int r, int lane) {
  typedef FragTr<D> __attribute__((aligned(4 * T32<D>::kMB))) aligned_frag;
  return *reinterpret_cast<const aligned_frag*>(tile + crow(r, lane >> 5) * T32<D>::kRS + T32<D>::kMB * (lane & 31));
}

// X . B^T over the columns: C rows = tile rows, C columns = the rows held in `b`
template <int D, int N>
__device__ __forceinline__ f32x16 product_rm(const float* tile, const f32x4v (&b)[T32<D>::kC], int lane) {
  f32x16 s[N];
#pragma unroll
  for (int i = 0; i < N; ++i) s[i] = zero16();
#pragma unroll
  for (int c = 0; c < T32<D>::kC; ++c) {
    const f32x4v a = frag_rm<D>(tile, c, lane);
#pragma unroll
    for (int i = 0; i < 4; ++i) s[i % N] = mfma(a[i], b[c][i], s[i % N]);
  }
  return add_chains(s);
}
// the same with both operands read from LDS
template <int D, int N>
__device__ __forceinline__ f32x16 product_rm2(const float* tile, const float* btile, int lane) {
  f32x16 s[N];
#pragma unroll
  for (int i = 0; i < N; ++i) s[i] = zero16();
#pragma unroll
  for (int c = 0; c < T32<D>::kC; ++c) {
    const f32x4v a = frag_rm<D>(tile, c, lane), b = frag_rm<D>(btile, c, lane);
#pragma unroll
    for (int i = 0; i < 4; ++i) s[i % N] = mfma(a[i], b[i], s[i % N]);
  }
  return add_chains(s);
}
// acc[column][.] += tile^T . w over the rows
template <int D>
__device__ __forceinline__ void product_tr(const float* tile, const f32x16& w, f32x16 (&acc)[T32<D>::kMB], int lane) {
#pragma unroll
  for (int r = 0; r < 16; ++r) {
    const FragTr<D> a = frag_tr<D>(tile, r, lane);
#pragma unroll
    for (int mb = 0; mb < T32<D>::kMB; ++mb) acc[mb] = mfma(a.v[mb], w[r], acc[mb]);
  }
}
// an accumulator of product_tr (lane = row, registers = columns) back into a row-major tile
template <int D>
__device__ __forceinline__ void put_rows(float* tile, const f32x16 (&acc)[T32<D>::kMB], int lane) {
  constexpr int MB = T32<D>::kMB;
  float* row = tile + (lane & 31) * T32<D>::kRS;
#pragma unroll
  for (int q = 0; q < 4; ++q) {  // C rows 8q + 4hh .. + 3: columns MB (8q + 4hh) .. + 4 MB - 1
#pragma unroll
    for (int k = 0; k < MB; ++k) {
      f32x4v v;
#pragma unroll
      for (int e = 0; e < 4; ++e) {
        const int col = 4 * k + e;
        v[e] = acc[col % MB][4 * q + col / MB];
      }
      *reinterpret_cast<f32x4v*>(row + MB * (8 * q + 4 * (lane >> 5)) + 4 * k) = v;
    }
  }
}
// sum over the four waves' tiles of one 16-byte piece of a row
template <int D>
__device__ __forceinline__ f32x4v sum_waves(const float* tiles, int wave_stride, int row, int part) {
  f32x4v t[kWaves];
#pragma unroll
  for (int w = 0; w < kWaves; ++w) t[w] = *reinterpret_cast<const f32x4v*>(tiles + w * wave_stride + row * T32<D>::kRS + 4 * part);
  return (t[0] + t[1]) + (t[2] + t[3]);
}

__device__ __forceinline__ float gate_logit(const segpt_attn_params& p, int b, int h, int row) {
  return reinterpret_cast<const float*>(p.gate.ptr)[(int64_t)b * p.gate.stride_b + (int64_t)row * p.gate.stride_s + (int64_t)h * p.gate.stride_h];
}

// ---- what follows the loops.  The four waves' results lie in `tiles`, `wave_stride` floats apart.

// forward: (maximum, sum, O) of the waves to y and lse
template <int D>
__device__ __forceinline__ void merge_waves(const segpt_attn_params& p, int b, int h, int q0, const float (*msm)[32], const float (*lsm)[32],
                                            const float* tiles, int wave_stride, int tid) {
  using T = T32<D>;
  const int part = tid % T::kLPR;
#pragma unroll
  for (int row = tid / T::kLPR; row < kRows; row += kThreads / T::kLPR) {
    float w[kWaves];
    const float M = fmaxf(fmaxf(msm[0][row], msm[1][row]), fmaxf(msm[2][row], msm[3][row]));
    float L = 0.f;
#pragma unroll
    for (int x = 0; x < kWaves; ++x) {
      w[x] = __builtin_amdgcn_exp2f(msm[x][row] - M);  // a wave without keys has (-inf, 0): weight 0
      L += lsm[x][row] * w[x];
    }
    f32x4v y = {0.f, 0.f, 0.f, 0.f};
#pragma unroll
    for (int x = 0; x < kWaves; ++x) {
      const f32x4v t = *reinterpret_cast<const f32x4v*>(tiles + x * wave_stride + row * T::kRS + 4 * part);
#pragma unroll
      for (int e = 0; e < 4; ++e) y[e] += w[x] * t[e];
    }
    if (q0 + row < p.Sq) {
      float f = 1.0f / L;
      if (p.gate.ptr) f *= p.gate_scale * sigmoidf_acc(gate_logit(p, b, h, q0 + row));
#pragma unroll
      for (int e = 0; e < 4; ++e) y[e] *= f;
      *reinterpret_cast<f32x4v*>(row_ptr_mut<float>(p.o, b, h, q0 + row) + 4 * part) = y;
      if (part == 0) p.lse[((int64_t)b * p.H + h) * p.Sq + q0 + row] = M * kLn2 + logf(L);
    }
  }
}

// dQ: T through the normaliser of q, and the workgroup's partial of the scale gradient, number part_row (red: kWaves * D floats of LDS)
template <int D>
__device__ __forceinline__ void finish_dq(const KArgs& a, int b, int h, int q0, int part_row, const float* tiles, int wave_stride, float* red, int tid) {
  const segpt_attn_params& p = a.p;
  using T = T32<D>;
  const int lane = tid & 63, wave = __builtin_amdgcn_readfirstlane(tid >> 6);
  // ---- through the q normaliser, u = dL/d(a q) = sm_scale g T; q is read again (its rotated form is what was normalised)
  const int part = tid % T::kLPR;
  f32x4v dg = {0.f, 0.f, 0.f, 0.f}, gl;
#pragma unroll
  for (int e = 0; e < 4; ++e) gl[e] = gprod<D>(p, 4 * part + e) * p.sm_scale;
#pragma unroll
  for (int row = tid / T::kLPR; row < kRows; row += kThreads / T::kLPR) {
    const bool live = q0 + row < p.Sq;
    const int rc = live ? q0 + row : p.Sq - 1;
    f32x4v q = *reinterpret_cast<const f32x4v*>(row_ptr<float>(p.q, b, h, rc) + 4 * part);
    if (p.rope_cos) q = rope_row<D, false>(p, q, p.rope_q_pos0 + rc, part);
    const float alpha = row_normaliser(p, row_sum<T::kLPR>((q[0] * q[0] + q[1] * q[1]) + (q[2] * q[2] + q[3] * q[3])), 1.0f / D);
    const f32x4v tt = sum_waves<D>(tiles, wave_stride, row, part);
    f32x4v u, dq;
    float dot = 0.f;
#pragma unroll
    for (int e = 0; e < 4; ++e) {
      u[e] = gl[e] * tt[e];
      dot += u[e] * q[e];
      dg[e] += live ? p.sm_scale * alpha * q[e] * tt[e] : 0.f;
    }
    const float a3 = norm_grad_coef(p, alpha, 1.0f / D) * row_sum<T::kLPR>(dot);
#pragma unroll
    for (int e = 0; e < 4; ++e) dq[e] = alpha * u[e] - a3 * q[e];
    if (p.rope_cos) dq = rope_row<D, true>(p, dq, p.rope_q_pos0 + rc, part);
    if (live) *reinterpret_cast<f32x4v*>(row_ptr_mut<float>(p.dq, b, h, rc) + 4 * part) = dq;
  }
  // the workgroup's rows of dg: over the rows of a wave, then over the waves
#pragma unroll
  for (int e = 0; e < 4; ++e)
#pragma unroll
    for (int o = T::kLPR; o < 64; o <<= 1) dg[e] += __shfl_xor(dg[e], o, 64);
  if (lane < T::kLPR) *reinterpret_cast<f32x4v*>(red + wave * D + 4 * lane) = dg;
  __syncthreads();
  if (tid < D) a.dg_part[(int64_t)part_row * D + tid] = (red[tid] + red[D + tid]) + (red[2 * D + tid] + red[3 * D + tid]);
}

}  // namespace
}  // namespace segpt
