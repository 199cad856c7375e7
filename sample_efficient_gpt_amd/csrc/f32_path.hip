// fp32 path: flash attention with fused QK-norm, forward and backward, on the fp32 matrix instruction
// v_mfma_f32_32x32x2_f32 (fp32 operands, fp32 accumulation).
//
// What bounds it: the fp32 matrix pipe (157 TFLOP/s, a sixteenth of bf16's).  One 32x32 block of scores at head_dim 64
// is 32 matrix instructions of 64 cycles per product, so LDS reads, exponentials and the row arithmetic hide behind it
// as soon as two waves share a SIMD; what has to be got right is keeping every SIMD busy:
//   * work unit = 32 rows of the stationary operand per WORKGROUP, and the four waves of a workgroup split the
//     STREAMED rows (wave w takes the 32-row tiles w, w + 4, ...).  The usual split (waves own different stationary
//     rows) needs 128 rows per workgroup: 128 workgroups at B = 2, H = 8, S = 1000, half the card.
//   * a wave stages its own tiles in its own LDS region: no workgroup barrier in the loop, the next tile's rows travel
//     in registers while the current one is computed.
//   * the four waves' results are merged once, through the same LDS, behind the loop.
// Measured at B = 2, H = 8, Hkv = 4, S = 1000, D = 64, against kernels of plain FMAs over 64-row workgroups: forward
// 385 -> 32 us, dQ 339 -> 43 us, dK/dV 787 -> 66 us.  With the card full (B = 8, H = 18, Hkv = 6, S = 2048): 94 / 102 /
// 99 TFLOP/s executed, 60-65 % of the pipe; the rest is the staging arithmetic (about 500 vector instructions per tile
// beside 64 to 128 matrix instructions) and LDS latency that two waves per SIMD do not cover entirely.
//
// Operand layouts of v_mfma_f32_32x32x2_f32 (hh = lane / 32): A: row = lane % 32, k = hh; B: column = lane % 32, k = hh;
// C: column = lane % 32, row(r) = 8 (r / 4) + 4 hh + r % 4.  The contraction order is free as long as both operands
// agree, and so is the order of the output rows, which gives two fragment reads of a row-major tile:
//   rm  (contraction over the columns): lane reads columns 8 c + 4 hh .. + 3 of row lane % 32 as one 16-byte read; its
//       four values are the k = hh entries of four matrix instructions.
//   tr  (contraction over the rows): register r of a C tile holds row row(r), so it IS the B operand of the instruction
//       that contracts the rows {row(r) at hh = 0, row(r) at hh = 1}; the lane reads the MB = D / 32 columns
//       MB (lane % 32) .. of that row, output row i of block mb then stands for column MB i + mb.
#include "common.hpp"

namespace segpt {

int f32_dq_grid(const segpt_attn_params& p);

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

// Work items are listed heaviest first.  When the whole grid is resident at once (up to two workgroups on each of 256
// CUs) or nearly so, the CU that got item i also gets item i + 256: every second round of 256 is dealt in reverse, so
// that a heavy item shares its CU with a light one (512 items: forward 37.8 -> 31.8 us, dQ 51 -> 43).  Larger grids
// balance by themselves and keep the plain order (dK/dV 3 % slower reversed at 9216 items).
__device__ __forceinline__ int work_item() {
  const int id = blockIdx.x, n = gridDim.x, round = id >> 8;
  if (n > 1024 || !(round & 1)) return id;
  return min((round << 8) + 255, n - 1) - (id & 255);
}

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
// side by side, and the one branch (rotary tables or not) stands outside the row loop.
template <int D, bool TINY_EPS>
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
    *reinterpret_cast<f32x4v*>(tile + (ps * T::kRPP + lr) * T::kRS + 4 * part) = x[ps] * (n * scale);
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

// ---- forward.  S^T = Khat Qhat^T (lane = query), running maximum per lane, O^T += V'^T P^T; every wave has its own
// (maximum, sum, O) over its keys, merged behind the loop.  Grid: heaviest query tiles first.
template <int D, bool TINY_EPS>
__global__ __launch_bounds__(kThreads, T32<D>::kOcc) void fwd_f32_kernel(KArgs a) {
  const segpt_attn_params& p = a.p;
  using T = T32<D>;
  __shared__ __attribute__((aligned(16))) float tiles[kWaves][2][T::kTile];
  __shared__ float msm[kWaves][32], lsm[kWaves][32];
  const int tid = threadIdx.x, lane = tid & 63;
  const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
  const int ln = lane & 31, hh = lane >> 5;
  const int n_qt = (p.Sq + kRows - 1) / kRows, heads = p.B * p.H;
  const int item = work_item();
  const int qt = n_qt - 1 - item / heads, hb = item % heads;
  const int b = hb / p.H, h = hb % p.H, g = h / (p.H / p.Hkv);
  const int q0 = qt * kRows;
  float c1 = 1.f, c2 = 0.f;
  if (p.vr_coef) { c1 = p.vr_coef[0]; c2 = p.vr_coef[1]; }
  float* kt = tiles[wave][0];
  float* vt = tiles[wave][1];

  int kend = p.Sk;
  if (p.causal) kend = min(p.Sk, q0 + kRows + p.q_start);
  const int n_kt = (kend + kRows - 1) / kRows;
  const float* kbase = row_ptr<float>(p.k, b, g, 0);
  f32x4v kraw[T::kPasses], vraw[T::kPasses], qraw[T::kPasses];
  load_tile<D>(qraw, row_ptr<float>(p.q, b, h, 0), p.q.stride_s, q0, p.Sq, lane);
  if (wave < n_kt) {
    load_tile<D>(kraw, kbase, p.k.stride_s, wave * kRows, p.Sk, lane);
    load_vmix<D>(p, vraw, b, g, wave * kRows, c1, c2, lane);
  }
  f32x4v one, gs;
#pragma unroll
  for (int e = 0; e < 4; ++e) {
    one[e] = 1.f;
    gs[e] = gprod<D>(p, 4 * (lane % T::kLPR) + e) * p.sm_scale * kLog2e;
  }
  f32x4v qf[T::kC];
  stage_norm<D, TINY_EPS>(p, qraw, gs, p.rope_q_pos0 + q0, p.Sq - 1 - q0, kt, lane);
  wave_sync();
#pragma unroll
  for (int c = 0; c < T::kC; ++c) qf[c] = frag_rm<D>(kt, c, lane);
  wave_sync();

  f32x16 o[T::kMB];
#pragma unroll
  for (int mb = 0; mb < T::kMB; ++mb) o[mb] = zero16();
  float m = -INFINITY, l = 0.f;  // l: this lane's half of the keys
  const int qlim = p.causal ? min(q0 + ln + p.q_start, p.Sk - 1) : p.Sk - 1;  // last visible key
  const int n_full = p.causal ? min(p.Sk, q0 + p.q_start + 1) / kRows : p.Sk / kRows;  // tiles that need no mask

  for (int jt = wave; jt < n_kt; jt += kWaves) {
    stage_norm<D, TINY_EPS>(p, kraw, one, p.rope_k_pos0 + jt * kRows, p.Sk - 1 - jt * kRows, kt, lane);
    stage_plain<D>(vraw, vt, lane);
    wave_sync();
    if (jt + kWaves < n_kt) {
      load_tile<D>(kraw, kbase, p.k.stride_s, (jt + kWaves) * kRows, p.Sk, lane);
      load_vmix<D>(p, vraw, b, g, (jt + kWaves) * kRows, c1, c2, lane);
    }
    f32x16 s = product_rm<D, 4>(kt, qf, lane);
    if (jt >= n_full) {
#pragma unroll
      for (int r = 0; r < 16; ++r)
        if (jt * kRows + crow(r, hh) > qlim) s[r] = -INFINITY;
    }
    float mx = s[0];
#pragma unroll
    for (int r = 1; r < 16; ++r) mx = fmaxf(mx, s[r]);
    mx = fmaxf(m, half_max(mx));
    const float mu = mx == -INFINITY ? 0.f : mx;
    if (__builtin_amdgcn_ballot_w64(mx > m) != 0) {  // some row has a new maximum
      const float corr = __builtin_amdgcn_exp2f(m - mu);
      l *= corr;
#pragma unroll
      for (int mb = 0; mb < T::kMB; ++mb)
#pragma unroll
        for (int r = 0; r < 16; ++r) o[mb][r] *= corr;
      m = mx;
    }
    float part[2] = {0.f, 0.f};
#pragma unroll
    for (int r = 0; r < 16; ++r) {
      s[r] = __builtin_amdgcn_exp2f(s[r] - mu);
      part[r & 1] += s[r];
    }
    l += part[0] + part[1];
    product_tr<D>(vt, s, o, lane);
    wave_sync();
  }

  // ---- merge the four waves
  const float lt = half_sum(l);
  if (hh == 0) { msm[wave][ln] = m; lsm[wave][ln] = lt; }
  put_rows<D>(kt, o, lane);
  __syncthreads();
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
      const f32x4v t = *reinterpret_cast<const f32x4v*>(&tiles[x][0][row * T::kRS + 4 * part]);
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

// ---- dQ: same split.  S^T and dP^T (lane = query), T^T += Khat^T dS^T.  Also owns everything per query row: delta =
// rowsum(dY o Y) (Y is the saved, already gated output, so this equals rowsum(dO o O)), dgate = (1 - sigmoid(z)) delta,
// the gate-scaled dO,
// and the workgroup's partial of the combined scale gradient  dg[d] = sum_i sm_scale (a_i q_id) T_id.
template <int D, bool TINY_EPS>
__global__ __launch_bounds__(kThreads, T32<D>::kOcc) void bwd_dq_f32_kernel(KArgs a) {
  const segpt_attn_params& p = a.p;
  using T = T32<D>;
  // four sums where the registers allow it (at head_dim 64 they spill): dq's distance to float64 at head_dim 128 3.6e-7 -> 3.0e-7,
  // step of 4 heads, 700 tokens 155.9 -> 156.6 us
  constexpr int kSums = D == 64 ? 2 : 4;
  __shared__ __attribute__((aligned(16))) float tiles[kWaves][2][T::kTile];
  __shared__ __attribute__((aligned(16))) float red[kWaves * D];
  __shared__ float dsm[kWaves][32];
  const int tid = threadIdx.x, lane = tid & 63;
  const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
  const int ln = lane & 31, hh = lane >> 5;
  const int n_qt = (p.Sq + kRows - 1) / kRows, heads = p.B * p.H;
  const int item = work_item();
  const int qt = n_qt - 1 - item / heads, hb = item % heads;
  const int b = hb / p.H, h = hb % p.H, g = h / (p.H / p.Hkv);
  const int q0 = qt * kRows;
  float c1 = 1.f, c2 = 0.f;
  if (p.vr_coef) { c1 = p.vr_coef[0]; c2 = p.vr_coef[1]; }
  float* kt = tiles[wave][0];
  float* vt = tiles[wave][1];
  const int64_t row_base = ((int64_t)b * p.H + h) * p.Sq;

  int kend = p.Sk;
  if (p.causal) kend = min(p.Sk, q0 + kRows + p.q_start);
  const int n_kt = (kend + kRows - 1) / kRows;
  const float* kbase = row_ptr<float>(p.k, b, g, 0);
  f32x4v gs;
#pragma unroll
  for (int e = 0; e < 4; ++e) gs[e] = gprod<D>(p, 4 * (lane % T::kLPR) + e) * p.sm_scale * kLog2e;
  f32x4v qf[T::kC], df[T::kC];
  {
    f32x4v x[T::kPasses], dy[T::kPasses], y[T::kPasses];
    load_tile<D>(x, row_ptr<float>(p.q, b, h, 0), p.q.stride_s, q0, p.Sq, lane);
    load_tile<D>(dy, row_ptr<float>(p.d_o, b, h, 0), p.d_o.stride_s, q0, p.Sq, lane);
    load_tile<D>(y, row_ptr<float>(p.o, b, h, 0), p.o.stride_s, q0, p.Sq, lane);
    stage_norm<D, TINY_EPS>(p, x, gs, p.rope_q_pos0 + q0, p.Sq - 1 - q0, kt, lane);
#pragma unroll
    for (int ps = 0; ps < T::kPasses; ++ps) {
      const int row = ps * T::kRPP + lane / T::kLPR;
      const f32x4v t = dy[ps] * y[ps];
      const float delta = row_sum<T::kLPR>((t[0] + t[1]) + (t[2] + t[3]));
      float f = 1.f;
      if (p.gate.ptr) {
        const float sg = sigmoidf_acc(gate_logit(p, b, h, min(q0 + row, p.Sq - 1)));
        f = p.gate_scale * sg;
        if (wave == 0 && lane % T::kLPR == 0 && q0 + row < p.Sq)
          reinterpret_cast<float*>(p.dgate.ptr)[(int64_t)b * p.dgate.stride_b + (int64_t)(q0 + row) * p.dgate.stride_s + (int64_t)h * p.dgate.stride_h] = (1.0f - sg) * delta;
      }
      if (lane % T::kLPR == 0) {
        dsm[wave][row] = delta;
        if (wave == 0 && q0 + row < p.Sq) a.delta[row_base + q0 + row] = delta;
      }
      dy[ps] *= f;
      if (a.do_eff && wave == 0 && q0 + row < p.Sq)  // gated: the copy the dK/dV kernel streams
        *reinterpret_cast<f32x4v*>(reinterpret_cast<float*>(a.do_eff) + (row_base + q0 + row) * D + 4 * (lane % T::kLPR)) = dy[ps];
    }
    stage_plain<D>(dy, vt, lane);
  }
  wave_sync();
#pragma unroll
  for (int c = 0; c < T::kC; ++c) {
    qf[c] = frag_rm<D>(kt, c, lane);
    df[c] = frag_rm<D>(vt, c, lane);
  }
  const float delta = dsm[wave][ln];
  const float lse = p.lse[row_base + min(q0 + ln, p.Sq - 1)];
  wave_sync();
  f32x4v kraw[T::kPasses], vraw[T::kPasses];
  if (wave < n_kt) {
    load_tile<D>(kraw, kbase, p.k.stride_s, wave * kRows, p.Sk, lane);
    load_vmix<D>(p, vraw, b, g, wave * kRows, c1, c2, lane);
  }
  f32x4v one;
#pragma unroll
  for (int e = 0; e < 4; ++e) one[e] = 1.f;
  f32x16 t[T::kMB];
#pragma unroll
  for (int mb = 0; mb < T::kMB; ++mb) t[mb] = zero16();
  const int qlim = p.causal ? min(q0 + ln + p.q_start, p.Sk - 1) : p.Sk - 1;
  const int n_full = p.causal ? min(p.Sk, q0 + p.q_start + 1) / kRows : p.Sk / kRows;

  for (int jt = wave; jt < n_kt; jt += kWaves) {
    stage_norm<D, TINY_EPS>(p, kraw, one, p.rope_k_pos0 + jt * kRows, p.Sk - 1 - jt * kRows, kt, lane);
    stage_plain<D>(vraw, vt, lane);
    wave_sync();
    if (jt + kWaves < n_kt) {
      load_tile<D>(kraw, kbase, p.k.stride_s, (jt + kWaves) * kRows, p.Sk, lane);
      load_vmix<D>(p, vraw, b, g, (jt + kWaves) * kRows, c1, c2, lane);
    }
    f32x16 s = product_rm<D, kSums>(kt, qf, lane);
    const f32x16 dp = product_rm<D, kSums>(vt, df, lane);
#pragma unroll
    for (int r = 0; r < 16; ++r) s[r] = prob(s[r], lse);
    if (jt >= n_full) {
#pragma unroll
      for (int r = 0; r < 16; ++r)
        if (jt * kRows + crow(r, hh) > qlim) s[r] = 0.f;
    }
#pragma unroll
    for (int r = 0; r < 16; ++r) s[r] *= dp[r] - delta;
    product_tr<D>(kt, s, t, lane);
    wave_sync();
  }

  put_rows<D>(kt, t, lane);
  __syncthreads();
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
    const f32x4v tt = sum_waves<D>(tiles[0][0], 2 * T::kTile, row, part);
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
  if (tid < D) a.dg_part[(int64_t)blockIdx.x * D + tid] = (red[tid] + red[D + tid]) + (red[2 * D + tid] + red[3 * D + tid]);
}

// ---- dK, dV of one query head: 32 keys stationary, query tiles streamed (Qhat and the gated dO).  S = Qhat Khat^T and
// dP = dO V'^T (lane = key), dV^T += dO^T P, dK^T += Qhat^T dS.  A workgroup takes every f32_splits-th group of four
// query tiles and writes its sums to the workspace; the finish kernel adds them over the query heads of the GQA group
// and the splits.  One workgroup per (key tile, KV head) walking all its query heads would leave the card half empty
// at small batches and its heaviest workgroup (first keys, every query) alone at the end.
template <int D, bool TINY_EPS>
__global__ __launch_bounds__(kThreads, T32<D>::kOcc) void bwd_dkdv_f32_kernel(KArgs a) {
  const segpt_attn_params& p = a.p;
  using T = T32<D>;
  constexpr int kSums = D == 64 ? 1 : 2;  // at head_dim 64 two sums spill
  __shared__ __attribute__((aligned(16))) float tiles[kWaves][2][T::kTile];
  __shared__ __attribute__((aligned(16))) float vtile[T::kTile];  // V' of the 32 keys: 32 registers fewer than as fragments
  __shared__ __attribute__((aligned(16))) float stat[kWaves][2][32];
  const int tid = threadIdx.x, lane = tid & 63;
  const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
  const int ln = lane & 31, hh = lane >> 5;
  const int units = p.B * p.H * a.f32_splits;  // heaviest key tiles (the first ones) first
  const int item = work_item();
  const int kt_i = item / units;
  int rest = item % units;
  const int split = rest % a.f32_splits;
  rest /= a.f32_splits;
  const int b = rest / p.H, h = rest % p.H, g = h / (p.H / p.Hkv);
  const int j0 = kt_i * kRows;
  float* qt = tiles[wave][0];
  float* dt = tiles[wave][1];
  const int64_t row_base = ((int64_t)b * p.H + h) * p.Sq;

  f32x4v one, gs;
#pragma unroll
  for (int e = 0; e < 4; ++e) {
    one[e] = 1.f;
    gs[e] = gprod<D>(p, 4 * (lane % T::kLPR) + e) * p.sm_scale * kLog2e;
  }
  f32x4v kf[T::kC];
  {
    float c1 = 1.f, c2 = 0.f;
    if (p.vr_coef) { c1 = p.vr_coef[0]; c2 = p.vr_coef[1]; }
    f32x4v k[T::kPasses], v[T::kPasses];
    load_tile<D>(k, row_ptr<float>(p.k, b, g, 0), p.k.stride_s, j0, p.Sk, lane);
    if (wave == 0) load_vmix<D>(p, v, b, g, j0, c1, c2, lane);
    stage_norm<D, TINY_EPS>(p, k, one, p.rope_k_pos0 + j0, p.Sk - 1 - j0, qt, lane);
    if (wave == 0) stage_plain<D>(v, vtile, lane);
    __syncthreads();
#pragma unroll
    for (int c = 0; c < T::kC; ++c) kf[c] = frag_rm<D>(qt, c, lane);
    wave_sync();
  }

  const int n_it = (p.Sq + kRows - 1) / kRows;
  const int first = p.causal ? max(0, j0 - p.q_start) / kRows : 0;  // the first tile that holds a query seeing key j0
  const int step = kWaves * a.f32_splits;
  int it = first + split * kWaves + wave;
  const float* qbase = row_ptr<float>(p.q, b, h, 0);
  const float* dbase = a.do_eff ? reinterpret_cast<const float*>(a.do_eff) + row_base * D : row_ptr<float>(p.d_o, b, h, 0);
  const int64_t dstep = a.do_eff ? D : p.d_o.stride_s;
  f32x4v qraw[T::kPasses], draw[T::kPasses];
  float lse_l = 0.f, delta_l = 0.f;
  auto request = [&](int tile) {
    load_tile<D>(qraw, qbase, p.q.stride_s, tile * kRows, p.Sq, lane);
    load_tile<D>(draw, dbase, dstep, tile * kRows, p.Sq, lane);
    const int64_t ri = row_base + min(tile * kRows + ln, p.Sq - 1);
    lse_l = p.lse[ri];
    delta_l = a.delta[ri];
  };
  if (it < n_it) request(it);
  f32x16 dk[T::kMB], dv[T::kMB];
#pragma unroll
  for (int mb = 0; mb < T::kMB; ++mb) dk[mb] = dv[mb] = zero16();

  for (; it < n_it; it += step) {
    const int i0 = it * kRows;
    stage_norm<D, TINY_EPS>(p, qraw, gs, p.rope_q_pos0 + i0, p.Sq - 1 - i0, qt, lane);
    stage_plain<D>(draw, dt, lane);
    if (hh == 0) { stat[wave][0][ln] = lse_l; stat[wave][1][ln] = delta_l; }
    wave_sync();
    if (it + step < n_it) request(it + step);
    f32x16 s = product_rm<D, kSums>(qt, kf, lane);
    const f32x16 dp = product_rm2<D, kSums>(dt, vtile, lane);
#pragma unroll
    for (int q = 0; q < 4; ++q) {
      const f32x4v ls = *reinterpret_cast<const f32x4v*>(&stat[wave][0][8 * q + 4 * hh]);
#pragma unroll
      for (int e = 0; e < 4; ++e) s[4 * q + e] = prob(s[4 * q + e], ls[e]);
    }
    if (i0 + kRows > p.Sq || (p.causal && j0 + kRows - 1 > i0 + p.q_start)) {
#pragma unroll
      for (int r = 0; r < 16; ++r) {
        const int i = i0 + crow(r, hh);
        if (i >= p.Sq || (p.causal && j0 + ln > i + p.q_start)) s[r] = 0.f;
      }
    }
    product_tr<D>(dt, s, dv, lane);
#pragma unroll
    for (int q = 0; q < 4; ++q) {
      const f32x4v de = *reinterpret_cast<const f32x4v*>(&stat[wave][1][8 * q + 4 * hh]);
#pragma unroll
      for (int e = 0; e < 4; ++e) s[4 * q + e] *= dp[4 * q + e] - de[e];
    }
    product_tr<D>(qt, s, dk, lane);
    wave_sync();
  }

  put_rows<D>(qt, dk, lane);
  put_rows<D>(dt, dv, lane);
  __syncthreads();
  const int part = tid % T::kLPR;
  const int64_t out = (((int64_t)b * p.H + h) * a.f32_splits + split) * p.Sk * D;
#pragma unroll
  for (int row = tid / T::kLPR; row < kRows; row += kThreads / T::kLPR) {
    if (j0 + row >= p.Sk) continue;
    const int64_t at = out + (int64_t)(j0 + row) * D + 4 * part;
    *reinterpret_cast<f32x4v*>(a.f32_dk_part + at) = sum_waves<D>(tiles[0][0], 2 * T::kTile, row, part);
    *reinterpret_cast<f32x4v*>(a.f32_dv_part + at) = sum_waves<D>(tiles[0][1], 2 * T::kTile, row, part);
  }
}

// ---- sums the partials of dK/dV in a fixed order, takes dKhat through the normaliser (khat = b k; the scale vector
// lives in Qhat, which also carries log2 e), writes dk, dv (, dv_first and the workgroup's sums for d vr_coef).
// Workgroup 0 adds up the scale gradient instead.
template <int D>
__global__ __launch_bounds__(kThreads) void bwd_finish_f32_kernel(KArgs a) {
  const segpt_attn_params& p = a.p;
  using T = T32<D>;
  __shared__ float red[kThreads];
  __shared__ float tot[D];
  const int tid = threadIdx.x;
  if (blockIdx.x == 0) {
    reduce_scale_grad<kThreads>(a, tid, red, tot);
    return;
  }
  const int part = tid % T::kLPR;
  const int64_t nrows = (int64_t)p.B * p.Hkv * p.Sk;
  const int64_t rid = (int64_t)(blockIdx.x - 1) * (kThreads / T::kLPR) + tid / T::kLPR;
  const bool live = rid < nrows;
  const int64_t rr = live ? rid : nrows - 1;
  const int j = (int)(rr % p.Sk), g = (int)(rr / p.Sk % p.Hkv), b = (int)(rr / ((int64_t)p.Sk * p.Hkv));
  const int rep = p.H / p.Hkv, n_part = rep * a.f32_splits;
  const int64_t at = (((int64_t)b * p.H + (int64_t)g * rep) * a.f32_splits * p.Sk + j) * D + 4 * part;
  f32x4v k = *reinterpret_cast<const f32x4v*>(row_ptr<float>(p.k, b, g, j) + 4 * part);
  f32x4v w = {0.f, 0.f, 0.f, 0.f}, dv = {0.f, 0.f, 0.f, 0.f};
#pragma unroll 4
  for (int x = 0; x < n_part; ++x) {
    w += *reinterpret_cast<const f32x4v*>(a.f32_dk_part + at + (int64_t)x * p.Sk * D);
    dv += *reinterpret_cast<const f32x4v*>(a.f32_dv_part + at + (int64_t)x * p.Sk * D);
  }
  if (p.rope_cos) k = rope_row<D, false>(p, k, p.rope_k_pos0 + j, part);  // the normaliser saw the rotated row
  const float beta = row_normaliser(p, row_sum<T::kLPR>((k[0] * k[0] + k[1] * k[1]) + (k[2] * k[2] + k[3] * k[3])), 1.0f / D);
  float dot = 0.f;
#pragma unroll
  for (int e = 0; e < 4; ++e) {
    w[e] *= kLn2;
    dot += w[e] * k[e];
  }
  const float b3 = norm_grad_coef(p, beta, 1.0f / D) * row_sum<T::kLPR>(dot);
#pragma unroll
  for (int e = 0; e < 4; ++e) w[e] = beta * w[e] - b3 * k[e];
  if (p.rope_cos) w = rope_row<D, true>(p, w, p.rope_k_pos0 + j, part);
  float c1 = 1.f, c2 = 0.f, s1 = 0.f, s2 = 0.f;
  if (p.vr_coef) { c1 = p.vr_coef[0]; c2 = p.vr_coef[1]; }
  if (live) {
    *reinterpret_cast<f32x4v*>(row_ptr_mut<float>(p.dk, b, g, j) + 4 * part) = w;
    *reinterpret_cast<f32x4v*>(row_ptr_mut<float>(p.dv, b, g, j) + 4 * part) = c1 * dv;
    if (p.v_first.ptr) {
      *reinterpret_cast<f32x4v*>(row_ptr_mut<float>(p.dv_first, b, g, j) + 4 * part) = c2 * dv;
      const f32x4v v = *reinterpret_cast<const f32x4v*>(row_ptr<float>(p.v, b, g, j) + 4 * part);
      const f32x4v f = *reinterpret_cast<const f32x4v*>(row_ptr<float>(p.v_first, b, g, j) + 4 * part);
#pragma unroll
      for (int e = 0; e < 4; ++e) { s1 += dv[e] * v[e]; s2 += dv[e] * f[e]; }
    }
  }
  if (p.vr_coef) {
#pragma unroll
    for (int o = 1; o < 64; o <<= 1) { s1 += __shfl_xor(s1, o, 64); s2 += __shfl_xor(s2, o, 64); }
    if ((tid & 63) == 0) { red[(tid >> 6) * 2] = s1; red[(tid >> 6) * 2 + 1] = s2; }
    __syncthreads();
    if (tid < 2) a.dcoef_part[(int64_t)(blockIdx.x - 1) * 2 + tid] = (red[tid] + red[2 + tid]) + (red[4 + tid] + red[6 + tid]);
  }
}

template <int D, bool TINY_EPS>
int launch_fwd(const KArgs& a, hipStream_t st) {
  hipLaunchKernelGGL((fwd_f32_kernel<D, TINY_EPS>), dim3((unsigned)f32_dq_grid(a.p)), dim3(kThreads), 0, st, a);
  return (int)hipGetLastError();
}
template <int D, bool TINY_EPS>
int launch_dq(const KArgs& a, hipStream_t st) {
  hipLaunchKernelGGL((bwd_dq_f32_kernel<D, TINY_EPS>), dim3((unsigned)f32_dq_grid(a.p)), dim3(kThreads), 0, st, a);
  return (int)hipGetLastError();
}
template <int D, bool TINY_EPS>
int launch_dkdv(const KArgs& a, hipStream_t st) {
  const segpt_attn_params& p = a.p;
  const int n_kt = (p.Sk + kRows - 1) / kRows;
  hipLaunchKernelGGL((bwd_dkdv_f32_kernel<D, TINY_EPS>), dim3((unsigned)(n_kt * p.B * p.H * a.f32_splits)), dim3(kThreads), 0, st, a);
  const int rc = (int)hipGetLastError();
  if (rc) return rc;
  hipLaunchKernelGGL(bwd_finish_f32_kernel<D>, dim3((unsigned)(a.n_dkdv_blocks + 1)), dim3(kThreads), 0, st, a);
  return (int)hipGetLastError();
}

}  // namespace

int f32_dq_grid(const segpt_attn_params& p) { return ((p.Sq + kRows - 1) / kRows) * p.B * p.H; }
// workgroups of the finish kernel that own rows of dK (one more adds up the scale gradient)
int f32_finish_grid(const segpt_attn_params& p) {
  return (int)(((int64_t)p.B * p.Hkv * p.Sk * p.D + kFinishFloats - 1) / kFinishFloats);
}
// Into how many workgroups the query tiles of one (key tile, query head) are dealt: enough for two resident rounds of
// the card (2 workgroups on each of 256 CUs), as long as every wave keeps at least one tile.
int f32_dkdv_splits(const segpt_attn_params& p) {
  const int64_t units = (int64_t)((p.Sk + kRows - 1) / kRows) * p.B * p.H;
  const int want = (int)((1024 + units - 1) / units);
  const int most = ((p.Sq + kRows - 1) / kRows + kWaves - 1) / kWaves;
  return want < most ? (want > 0 ? want : 1) : most;
}

int launch_fwd_f32(const KArgs& a, hipStream_t st) {
  const bool tiny = tiny_eps(a.p);
  switch (a.p.D) {
    case 32: return tiny ? launch_fwd<32, true>(a, st) : launch_fwd<32, false>(a, st);
    case 64: return tiny ? launch_fwd<64, true>(a, st) : launch_fwd<64, false>(a, st);
    case 128: return tiny ? launch_fwd<128, true>(a, st) : launch_fwd<128, false>(a, st);
    default: return (int)hipErrorInvalidValue;
  }
}

int launch_bwd_dq_f32(const KArgs& a, hipStream_t st) {
  const bool tiny = tiny_eps(a.p);
  switch (a.p.D) {
    case 32: return tiny ? launch_dq<32, true>(a, st) : launch_dq<32, false>(a, st);
    case 64: return tiny ? launch_dq<64, true>(a, st) : launch_dq<64, false>(a, st);
    case 128: return tiny ? launch_dq<128, true>(a, st) : launch_dq<128, false>(a, st);
    default: return (int)hipErrorInvalidValue;
  }
}

int launch_bwd_dkdv_f32(const KArgs& a, hipStream_t st) {
  const bool tiny = tiny_eps(a.p);
  switch (a.p.D) {
    case 32: return tiny ? launch_dkdv<32, true>(a, st) : launch_dkdv<32, false>(a, st);
    case 64: return tiny ? launch_dkdv<64, true>(a, st) : launch_dkdv<64, false>(a, st);
    case 128: return tiny ? launch_dkdv<128, true>(a, st) : launch_dkdv<128, false>(a, st);
    default: return (int)hipErrorInvalidValue;
  }
}

}  // namespace segpt
