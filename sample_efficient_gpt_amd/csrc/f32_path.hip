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
#include "f32_common.hpp"

namespace segpt {
namespace {

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
  const int item = work_item(blockIdx.x, gridDim.x);
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
  merge_waves<D>(p, b, h, q0, msm, lsm, tiles[0][0], 2 * T::kTile, tid);
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
  const int item = work_item(blockIdx.x, gridDim.x);
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
  finish_dq<D>(a, b, h, q0, blockIdx.x, tiles[0][0], 2 * T::kTile, red, tid);
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
  const int item = work_item(blockIdx.x, gridDim.x);
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
    if (!a.f32_split || a.f32_both) reduce_scale_grad<kThreads>(a, tid, red, tot);  // else the other dK/dV kernel has done it
    return;
  }
  const int part = tid % T::kLPR;
  const int64_t nrows = (int64_t)p.B * p.Hkv * p.Sk;
  const int64_t rid = (int64_t)(blockIdx.x - 1) * (kThreads / T::kLPR) + tid / T::kLPR;
  const bool live = rid < nrows;
  const int64_t rr = live ? rid : nrows - 1;
  const int j = (int)(rr % p.Sk), g = (int)(rr / p.Sk % p.Hkv), b = (int)(rr / ((int64_t)p.Sk * p.Hkv));
  const int n_part = a.f32_parts;
  const int64_t at = (((int64_t)b * p.Hkv + g) * n_part * p.Sk + j) * D + 4 * part;
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
  return rc ? rc : launch_finish_f32(a, st);
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

int launch_finish_f32(const KArgs& a, hipStream_t st) {
  const dim3 grid((unsigned)(a.n_dkdv_blocks + 1)), block(kThreads);
  switch (a.p.D) {
    case 32: hipLaunchKernelGGL(bwd_finish_f32_kernel<32>, grid, block, 0, st, a); break;
    case 64: hipLaunchKernelGGL(bwd_finish_f32_kernel<64>, grid, block, 0, st, a); break;
    case 128: hipLaunchKernelGGL(bwd_finish_f32_kernel<128>, grid, block, 0, st, a); break;
    default: return (int)hipErrorInvalidValue;
  }
  return (int)hipGetLastError();
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
