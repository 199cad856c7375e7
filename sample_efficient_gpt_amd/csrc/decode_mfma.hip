// bf16 forward for decode-shaped calls: a handful of query rows (H/Hkv * Sq <= 32 per kv head) against a long
// key/value cache (the reference's generation path: attention.py:191-198 builds q_start = past length,
// KVCache :15-27 grows K/V, the module masks with k_idx <= q_start + q_idx, :72-78).
//
// The training kernel would run B*H workgroups that each walk the whole cache; here the KEYS are split
// ("flash decoding"): wave (b, kv head g, split s) handles one contiguous chunk of the cache for ALL query
// rows of the group (n = hq * Sq + i, at most 32 = one MFMA column block), writes an unnormalised partial
// (running maximum M, sum L, O) and a second tiny kernel merges the splits.  Memory-bound by design: every
// K / V row is read exactly once from HBM, so the key normalisation, the rotary embedding and the value
// residual mix are done on the fly in registers (no pre-pass, no normalised copy).
//
// Per wave and 32-key block (orientation as in the training forward: lane = query column):
//   K rows from LDS in the MFMA A layout (row = key, 16-byte chunks), rotated if asked     S^T = K . Qhat^T  (4 or 8 MFMAs)
//   scores times b_j = rsqrt(mean k^2 + eps), exp2, P^T packed to bf16 = B operand
//   V rows by transposing LDS reads                                                        O^T += V'^T . P^T
#include <algorithm>

#include "mfma_common.hpp"

namespace segpt {
namespace {

constexpr int kDecThreads = 256;  // 4 waves
constexpr int kDecBlock = 32;     // keys per step of a wave
constexpr int kMaxSplits = 128;

// LDS regions below are private to a wave: program order is enough, the compiler only has to keep it
__device__ __forceinline__ void wave_lds_sync() {
  __builtin_amdgcn_fence(__ATOMIC_ACQ_REL, "wavefront");
  __builtin_amdgcn_wave_barrier();
}

// acc + lo^2 + hi^2 of a packed bf16 pair (fp32 products and sum)
__device__ __forceinline__ float sum_sq_bf16_pair(uint32_t w, float acc) {
  typedef __bf16 bf2 __attribute__((ext_vector_type(2)));
  const bf2 v = __builtin_bit_cast(bf2, w);
  return __builtin_amdgcn_fdot2_f32_bf16(v, v, acc, false);
}

// One 32-row tile filled by ONE wave (swizzled like every tile of Swz): lane offsets of its wave-wide loads from the
// tile's first row; rows past rows_left re-read the last one.
template <int D>
struct WaveTile {
  static constexpr int kLoads = Swz<D, kDecBlock>::kTileBytes / 1024;
  uint32_t off[kLoads];
};
template <int D>
__device__ __forceinline__ WaveTile<D> wave_tile_offsets(uint32_t step, int rows_left, int lane) {
  using Z = Swz<D, kDecBlock>;
  WaveTile<D> o;
#pragma unroll
  for (int i = 0; i < WaveTile<D>::kLoads; ++i) {
    const int row = i * Z::kRowsPerInst + lane / Z::kChunks;
    o.off[i] = (uint32_t)min(row, rows_left - 1) * step + (((lane % Z::kChunks) ^ Z::f(row)) << 4);
  }
  return o;
}
template <int D>
__device__ __forceinline__ void issue_wave_tile(const char* base, const WaveTile<D>& o, uint32_t dst) {
#pragma unroll
  for (int i = 0; i < WaveTile<D>::kLoads; ++i) gload_lds16_so(base, o.off[i], dst + i * 1024);
}
// this wave's LDS reads have returned (before the tile they came from is requested over)
__device__ __forceinline__ void wait_lds_reads() {
  wave_lds_sync();
  __builtin_amdgcn_s_waitcnt(0xC07F);  // lgkmcnt(0) only
}

// One wave per (batch, kv head, split).  The four waves of a workgroup take the SAME keys of four consecutive (batch, kv
// head) pairs, so that with a rotary embedding the table rows of a key block (as long as a K row each: cos and sin
// together as much as K and V) come in once per workgroup, double-buffered one block ahead.
//
// Bound by HBM: every K and V row once.  What the memory system needs for that is whole lines and requests that stay in
// flight, so K, V, V_first and the tables all travel by direct global->LDS loads into swizzled tiles (see the request
// order below).  Before, every lane loaded 16-byte pieces of its own row and, with a rotary embedding, of the two
// table rows, by each wave for itself.  B = 32, 6 kv heads, 8192 keys, head_dim 64 (403 MB): 121.7 -> 79.1 us with a
// rotary embedding, 83.8 -> 77.8 without; B = 8, 4 kv heads, 5001 keys, head_dim 128 (82 MB): 33.8 -> 22.9 us.  (Sharing
// the tables alone: 85.8 and 30.6 us.)
//
// What else keeps the loop near the memory rate (it has about 200 vector instructions per 32 keys to hide):
//   * the normaliser b_j multiplies the 16 scores a lane holds, not the 32 K entries: without a rotary embedding the raw
//     K bits ARE the matrix operand and the row's sum of squares is 16 dot instructions;
//   * no running maximum where the QK-norm bound on the logits allows none (see logit_bound), else a lazily raised one;
//   * only the block that holds the last visible key is masked;
//   * with a value residual c1 P and c2 P are the operands of two products, V and V_first the raw rows of both.
// Each wave writes its own partial (M, L, O) of its n_rows live query rows: nothing is merged inside the workgroup.
// workgroups per CU that LDS (tiles and tables) and registers allow
template <int D, bool ROPE, bool VRES>
constexpr int kDecOcc = D == 64 ? (VRES ? 2 : 3) : (ROPE || VRES ? 1 : 2);

template <int D, bool ROPE, bool VRES>
__global__ __launch_bounds__(kDecThreads, (kDecOcc<D, ROPE, VRES>)) void decode_split_kernel(KArgs a) {
  constexpr int KS = D / 16;
  constexpr int MB = D / 32;
  using Z = Swz<D, kDecBlock>;
  const segpt_attn_params& p = a.p;
  __shared__ __attribute__((aligned(1024))) char tab[ROPE ? 2 * 2 * Z::kTileBytes : 16];  // [buffer][cos, sin] of a key block
  __shared__ __attribute__((aligned(1024))) char tiles[4][VRES ? 3 : 2][Z::kTileBytes];  // wave-private K, V (, V_first) rows
  __shared__ __attribute__((aligned(16))) float bsm[4][kDecBlock];                  // wave-private b_j
  __shared__ __attribute__((aligned(16))) float gsm[D];

  const int tid = threadIdx.x, lane = tid & 63;
  const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
  const int ln = lane & 31, hh = lane >> 5;
  const int rep = p.H / p.Hkv;
  const int n_rows = rep * p.Sq;  // query rows of this kv head, <= 32
  const int split = blockIdx.x % a.dec_splits;
  const int bg_all = p.B * p.Hkv, bg_raw = 4 * (int)(blockIdx.x / a.dec_splits) + wave;
  const bool active = bg_raw < bg_all;  // wave-uniform; an idle wave of the last workgroup only keeps the barriers
  const int bg = active ? bg_raw : bg_all - 1;
  const int g = bg % p.Hkv, b = bg / p.Hkv;
  const int k_lo = split * a.dec_chunk;
  const int k_hi = min(k_lo + a.dec_chunk, a.dec_kend);

  const int2 src = swz_src<D>(lane, wave);
  const uint32_t tab0 = lds_addr_of(tab);
  auto issue_tables = [&](int jb, int buf) {
    const int64_t row0 = (int64_t)(p.rope_k_pos0 + jb) * (D / 2);
    issue_tile_pair<D, kDecBlock>(reinterpret_cast<const char*>(p.rope_cos + row0), reinterpret_cast<const char*>(p.rope_sin + row0),
                                  tile_lane_offsets<D, kDecBlock>(D * 2, D * 2, p.Sk - jb, src.x, src.y),
                                  tab0 + buf * 2 * Z::kTileBytes + wave * 1024);
  };
  if constexpr (ROPE) issue_tables(k_lo, 0);
  // Every row travels global -> LDS as part of whole lines (a row-per-lane load covers 32 bytes of each of 32 rows and
  // leaves the rest of their lines to the L1, which 64 KB in flight overrun).  One buffer per tensor: a tile is requested
  // again as soon as its last reader has its fragments, so K is in flight during the softmax and the V product, V during
  // the next block's scores.  Order of the requests: [tables, K, V, V_first] of block 0, then tables, K, V, V_first of
  // each next block; every wait below leaves exactly the younger ones in flight.
  constexpr int kTabLoads = ROPE ? 2 * Z::kPasses : 0, kRowLoads = WaveTile<D>::kLoads, kFirstLoads = VRES ? kRowLoads : 0;
  const char* kbase = reinterpret_cast<const char*>(row_ptr<uint16_t>(p.k, b, g, 0));
  const char* vbase = reinterpret_cast<const char*>(row_ptr<uint16_t>(p.v, b, g, 0));
  const char* fbase = VRES ? reinterpret_cast<const char*>(row_ptr<uint16_t>(p.v_first, b, g, 0)) : nullptr;
  const uint32_t kstep = (uint32_t)p.k.stride_s * 2, vstep = (uint32_t)p.v.stride_s * 2, fstep = (uint32_t)p.v_first.stride_s * 2;
  const uint32_t ktile = lds_addr_of(tiles[wave][0]), vtile = lds_addr_of(tiles[wave][1]), ftile = lds_addr_of(tiles[wave][VRES ? 2 : 1]);
  const WaveTile<D> koff = wave_tile_offsets<D>(kstep, kDecBlock, lane), voff = wave_tile_offsets<D>(vstep, kDecBlock, lane);
  auto issue_rows = [&](const char* base, uint32_t step, const WaveTile<D>& full, int jb, uint32_t dst) {
    const char* src = base + (int64_t)jb * step;
    if (p.Sk - jb >= kDecBlock) issue_wave_tile<D>(src, full, dst);
    else issue_wave_tile<D>(src, wave_tile_offsets<D>(step, p.Sk - jb, lane), dst);
  };
  auto issue_k = [&](int jb) { issue_rows(kbase, kstep, koff, jb, ktile); };
  auto issue_v = [&](int jb) { issue_rows(vbase, vstep, voff, jb, vtile); };
  auto issue_first = [&](int jb) {
    if constexpr (VRES) issue_wave_tile<D>(fbase + (int64_t)jb * fstep, wave_tile_offsets<D>(fstep, p.Sk - jb, lane), ftile);
  };
  if (active) {
    issue_k(k_lo);
    issue_v(k_lo);
    issue_first(k_lo);
  }

  // ---- this lane's query (B operand column n): Qhat = sm_scale*log2e * a q g_q g_k, zero for padding columns
  if (tid < D) gsm[tid] = gprod_at(p, tid) * p.sm_scale * kLog2e;
  __syncthreads();
  const bool bounded = !(p.flags & (SEGPT_FLAG_RUNNING_MAX | SEGPT_FLAG_NO_NORM)) && logit_bound<D>(gsm, lane) <= kNoMaxBound;  // wave-uniform
  const bool qlive = ln < n_rows;
  const int hq = qlive ? ln / p.Sq : 0, qi = qlive ? ln % p.Sq : 0;
  bf16x8 qreg[KS];
  {
    const uint16_t* qp = row_ptr<uint16_t>(p.q, b, g * rep + hq, qi) + 8 * hh;
    u32x4 raw[KS];
#pragma unroll
    for (int ks = 0; ks < KS; ++ks) raw[ks] = *reinterpret_cast<const u32x4*>(qp + 16 * ks);
    float x[KS][8];
    unpack_b_layout<KS>(raw, x);
    if constexpr (ROPE) {
      const int64_t pos = (int64_t)(p.rope_q_pos0 + qi) * (D / 2);
      rope_b_layout<KS>(x, p.rope_cos + pos, p.rope_sin + pos, hh);
    }
    float ss = 0.f;
#pragma unroll
    for (int ks = 0; ks < KS; ++ks)
#pragma unroll
      for (int t = 0; t < 8; ++t) ss += x[ks][t] * x[ks][t];
    ss = half_sum(ss);
    const float alpha = qlive ? row_normaliser_fast(p, ss, 1.0f / D) : 0.f;
#pragma unroll
    for (int ks = 0; ks < KS; ++ks) {
      const float4 ga = *reinterpret_cast<const float4*>(gsm + 16 * ks + 8 * hh);
      const float4 gb = *reinterpret_cast<const float4*>(gsm + 16 * ks + 8 * hh + 4);
      u32x4 w;
      w[0] = pack_bf16x2(x[ks][0] * alpha * ga.x, x[ks][1] * alpha * ga.y);
      w[1] = pack_bf16x2(x[ks][2] * alpha * ga.z, x[ks][3] * alpha * ga.w);
      w[2] = pack_bf16x2(x[ks][4] * alpha * gb.x, x[ks][5] * alpha * gb.y);
      w[3] = pack_bf16x2(x[ks][6] * alpha * gb.z, x[ks][7] * alpha * gb.w);
      qreg[ks] = as_bf16x8(w);
    }
  }
  // last visible key of this lane's query, and the last one every query row sees
  const int qlim = p.causal ? min(qi + p.q_start, p.Sk - 1) : p.Sk - 1;
  const int all_see = p.causal ? min(p.q_start, p.Sk - 1) : p.Sk - 1;

  float c1 = 1.f, c2 = 0.f;
  if constexpr (VRES) { c1 = p.vr_coef[0]; c2 = p.vr_coef[1]; }

  f32x16 oacc[MB];
#pragma unroll
  for (int mb = 0; mb < MB; ++mb) oacc[mb] = splat16(0.f);
  float m_ref = bounded ? 0.f : -INFINITY, l_run[2] = {0.f, 0.f};  // l_run: this lane's half of the keys, as two partial sums

  const uint32_t row16 = tab0 + swz_off_row16<D>(lane);
  const uint32_t krm = ktile + swz_off_rm<D>(lane), vtr = vtile + swz_off_tr<D>(lane), ftr = ftile + swz_off_tr<D>(lane);
  int buf = 0;
  wait_vmcnt<0>();  // nothing but tile requests may be in flight in the loop, whose waits count them
  wave_lds_sync();
  for (int jb = k_lo; jb < k_hi; jb += kDecBlock) {
    const bool more = jb + kDecBlock < k_hi;
    if (active) wait_vmcnt<kRowLoads + kFirstLoads>();  // this block's tables and K
    else wait_vmcnt<0>();
    if constexpr (ROPE) {
      __syncthreads();  // every wave's pieces of the tables are there, and nobody reads the other buffer any more
      if (more) issue_tables(jb + kDecBlock, buf ^ 1);
    }
    if (active) {
      wave_lds_sync();
      u32x4 kraw[KS];
#pragma unroll
      for (int ks = 0; ks < KS; ++ks) kraw[ks] = __builtin_bit_cast(u32x4, swz_frag_rm<D>(krm, 0, ks));
      float ss = 0.f;
      if constexpr (ROPE) {
        // one pair of 16-byte chunks (elements e and e + D/2) at a time: few registers beside the loads in flight
        const uint32_t cos16 = row16 + buf * 2 * Z::kTileBytes, sin16 = cos16 + Z::kTileBytes;
        float s4[4] = {0.f, 0.f, 0.f, 0.f};
#pragma unroll
        for (int ks = 0; ks < KS / 2; ++ks)
#pragma unroll
          for (int i = 0; i < 2; ++i) {
            const uint32_t off = (uint32_t)((4 * ks + 2 * hh + i) << 4);  // floats 16 ks + 8 hh + 4 i ..
            const f32x4 c = lds_read_f4(cos16 ^ off), sn = lds_read_f4(sin16 ^ off);
#pragma unroll
            for (int t = 0; t < 2; ++t) {
              const uint32_t wa = kraw[ks][2 * i + t], wb = kraw[ks + KS / 2][2 * i + t];
              float a0 = bf16lo(wa), a1 = bf16hi(wa), b0 = bf16lo(wb), b1 = bf16hi(wb);
              rope_pair(a0, b0, c[2 * t], sn[2 * t]);
              rope_pair(a1, b1, c[2 * t + 1], sn[2 * t + 1]);
              s4[0] += a0 * a0; s4[1] += a1 * a1; s4[2] += b0 * b0; s4[3] += b1 * b1;
              kraw[ks][2 * i + t] = pack_bf16x2(a0, a1);
              kraw[ks + KS / 2][2 * i + t] = pack_bf16x2(b0, b1);
            }
          }
        ss = (s4[0] + s4[1]) + (s4[2] + s4[3]);
      } else {
        float s2[2] = {0.f, 0.f};
#pragma unroll
        for (int ks = 0; ks < KS; ++ks)
#pragma unroll
          for (int i = 0; i < 4; ++i) s2[i & 1] = sum_sq_bf16_pair(kraw[ks][i], s2[i & 1]);
        ss = s2[0] + s2[1];
      }
      ss = half_sum(ss);
      if (hh == 0) bsm[wave][ln] = row_normaliser_fast(p, ss, 1.0f / D);
      f32x16 s = splat16(0.f);
#pragma unroll
      for (int ks = 0; ks < KS; ++ks) s = mfma32(as_bf16x8(kraw[ks]), qreg[ks], s);
      wait_lds_reads();
      if (more) issue_k(jb + kDecBlock);
      // register r holds key jb + 4hh + c_r, c_r = 8(r/4) + r%4
#pragma unroll
      for (int q = 0; q < 4; ++q) {
        const float4 bj = *reinterpret_cast<const float4*>(&bsm[wave][8 * q + 4 * hh]);
        s[4 * q + 0] *= bj.x; s[4 * q + 1] *= bj.y; s[4 * q + 2] *= bj.z; s[4 * q + 3] *= bj.w;
      }
      if (jb + kDecBlock - 1 > min(all_see, k_hi - 1)) {  // visible iff <= qlim and < k_hi
        const int t = min(qlim, k_hi - 1) - jb - 4 * hh;
#pragma unroll
        for (int r = 0; r < 16; ++r)
          if (8 * (r >> 2) + (r & 3) > t) s[r] = -INFINITY;
      }
      if (!bounded) {
        float mx = s[0];
#pragma unroll
        for (int r = 1; r < 16; ++r) mx = fmaxf(mx, s[r]);
        mx = half_max(mx);
        const bool need = mx > m_ref + kLazyThresh;
        if (__builtin_amdgcn_ballot_w64(need) != 0) {
          const float m_new = need ? mx : m_ref;
          const float corr = need ? fast_exp2(m_ref - m_new) : 1.0f;
          m_ref = m_new;
          l_run[0] *= corr;
          l_run[1] *= corr;
#pragma unroll
          for (int mb = 0; mb < MB; ++mb)
#pragma unroll
            for (int r = 0; r < 16; ++r) oacc[mb][r] *= corr;
        }
        const float mu = m_ref == -INFINITY ? 0.f : m_ref;  // nothing visible yet: keep exp2 away from inf - inf
#pragma unroll
        for (int r = 0; r < 16; ++r) s[r] -= mu;
      }
#pragma unroll
      for (int r = 0; r < 16; ++r) s[r] = fast_exp2(s[r]);
      auto add_product = [&](uint32_t tr, bf16x8 p0, bf16x8 p1) {
        wave_lds_sync();
#pragma unroll
        for (int mb = 0; mb < MB; ++mb) {
          oacc[mb] = mfma32(swz_frag_tr<D>(tr, mb, 0), p0, oacc[mb]);
          oacc[mb] = mfma32(swz_frag_tr<D>(tr, mb, 1), p1, oacc[mb]);
        }
        wait_lds_reads();
      };
      if (more) wait_vmcnt<kFirstLoads + kTabLoads + kRowLoads>(); else wait_vmcnt<kFirstLoads>();  // this block's V
      if constexpr (!VRES) {
        const bf16x8 p0 = pack_c_half_sum(s, 0, l_run), p1 = pack_c_half_sum(s, 1, l_run);
        add_product(vtr, p0, p1);
        if (more) issue_v(jb + kDecBlock);
      } else {
        f32x16 s1, s2;
#pragma unroll
        for (int r = 0; r < 16; ++r) {
          l_run[r & 1] += s[r];
          s1[r] = c1 * s[r];
          s2[r] = c2 * s[r];
        }
        add_product(vtr, pack_c_half(s1, 0), pack_c_half(s1, 1));
        if (more) { issue_v(jb + kDecBlock); wait_vmcnt<kTabLoads + 2 * kRowLoads>(); } else wait_vmcnt<0>();  // V_first
        add_product(ftr, pack_c_half(s2, 0), pack_c_half(s2, 1));
        if (more) issue_first(jb + kDecBlock);
      }
    }
    buf ^= 1;
  }

  // ---- this wave's partial: rows n of [bg, split][n_rows][D]
  const float l_tot = half_sum(l_run[0] + l_run[1]);
  if (active && qlive) {
    const int64_t at = ((int64_t)bg * a.dec_splits + split) * n_rows + ln;
#pragma unroll
    for (int mb = 0; mb < MB; ++mb)
#pragma unroll
      for (int q = 0; q < 4; ++q)
        *reinterpret_cast<float4*>(a.dec_part + at * D + 32 * mb + 8 * q + 4 * hh) =
            make_float4(oacc[mb][4 * q], oacc[mb][4 * q + 1], oacc[mb][4 * q + 2], oacc[mb][4 * q + 3]);
    if (hh == 0) *reinterpret_cast<float2*>(a.dec_stat + at * 2) = make_float2(m_ref, l_tot);
  }
}

// One workgroup per (batch, kv head, query row): merges the splits, normalises, gates, writes y (bf16) and lse
// (natural log).  Thread (group gi, column d) sums the splits gi, gi + G, ... of output column d (G = threads / D);
// its first partial values are requested before the split statistics are reduced, so that the kernel is about
// two memory round trips long whatever the number of splits.  Every sum has a fixed order: deterministic.
constexpr int kMergeThreads = 256;
constexpr int kMergeEarly = 16;  // partial values per thread requested up front

__global__ __launch_bounds__(kMergeThreads) void decode_merge_kernel(KArgs a) {
  const segpt_attn_params& p = a.p;
  __shared__ float wsm[kMaxSplits];
  __shared__ float redm[4], redl[4];
  __shared__ float part[kMergeThreads];
  const int D = p.D, tid = threadIdx.x, lane = tid & 63, wave = tid >> 6;
  const int rep = p.H / p.Hkv;
  const int n_rows = rep * p.Sq;
  const int n = blockIdx.x % n_rows, bg = blockIdx.x / n_rows;
  const int g = bg % p.Hkv, b = bg / p.Hkv;
  const int S = a.dec_splits;
  const int G = kMergeThreads / D, gi = tid / D, d = tid - gi * D;
  const float* col = a.dec_part + ((int64_t)bg * S * n_rows + n) * D + d;  // split sp: + sp * n_rows * D
  const float* ss = a.dec_stat + ((int64_t)bg * S * n_rows + n) * 2;
  const int64_t part_step = (int64_t)n_rows * D;
  float pv[kMergeEarly];
#pragma unroll
  for (int u = 0; u < kMergeEarly; ++u) {
    const int sp = gi + G * u;
    pv[u] = sp < S ? col[sp * part_step] : 0.f;
  }
  float m = -INFINITY;
  for (int sp = tid; sp < S; sp += kMergeThreads) m = fmaxf(m, ss[sp * n_rows * 2]);
#pragma unroll
  for (int o = 1; o < 64; o <<= 1) m = fmaxf(m, __shfl_xor(m, o, 64));
  if (lane == 0) redm[wave] = m;
  __syncthreads();
  const float M = fmaxf(fmaxf(redm[0], redm[1]), fmaxf(redm[2], redm[3]));
  float l = 0.f;
  for (int sp = tid; sp < S; sp += kMergeThreads) {
    const float w = exp2f(ss[sp * n_rows * 2] - M);  // a split with nothing visible has (-inf, 0): weight 0
    wsm[sp] = w;
    l += ss[sp * n_rows * 2 + 1] * w;
  }
#pragma unroll
  for (int o = 1; o < 64; o <<= 1) l += __shfl_xor(l, o, 64);
  if (lane == 0) redl[wave] = l;
  __syncthreads();  // also publishes wsm
  const float L = (redl[0] + redl[1]) + (redl[2] + redl[3]);
  float acc = 0.f;
#pragma unroll
  for (int u = 0; u < kMergeEarly; ++u) {
    const int sp = gi + G * u;
    if (sp < S) acc += pv[u] * wsm[sp];
  }
  for (int sp = gi + G * kMergeEarly; sp < S; sp += G) acc += col[sp * part_step] * wsm[sp];
  part[tid] = acc;
  __syncthreads();
  const int hq = n / p.Sq, qi = n % p.Sq;
  const int h = g * rep + hq;
  if (tid == 0) p.lse[((int64_t)b * p.H + h) * p.Sq + qi] = (M + log2f(L)) * kLn2;
  if (tid < D) {
    float f = 1.0f / L;
    if (p.gate.ptr) {
      const float z = bf16_to_f32(reinterpret_cast<const uint16_t*>(p.gate.ptr)[(int64_t)b * p.gate.stride_b + (int64_t)qi * p.gate.stride_s + (int64_t)h * p.gate.stride_h]);
      f *= p.gate_scale / (1.0f + __expf(-z));
    }
    float tot = part[tid];
    for (int x = 1; x < G; ++x) tot += part[x * D + tid];
    row_ptr_mut<uint16_t>(p.o, b, h, qi)[tid] = f32_to_bf16(tot * f);
  }
}

}  // namespace

// Split plan of a decode-shaped call: keys [0, kend) in `splits` chunks of `chunk` keys (whole 32-key blocks), no empty
// split.  One workgroup (four (batch, kv head) pairs) per CU already keeps 32 KB (head_dim 128: 64 KB) of rows in
// flight, and more of them only shorten the chunks: 8 x 4 pairs, 5001 keys, head_dim 128: 256 workgroups 22.9 us, 424
// 31.6, 632 38.5; 24 x 6 pairs, 1332 keys, head_dim 64: 252 workgroups 19.8 us, 756 23.1.  So the split count is the one
// that leaves the fewest blocks on the fullest CU with one workgroup on each; a second or third round only where it evens
// the load out by more than 3 % each (32 x 6 pairs, 8192 keys: 768 workgroups of 16 blocks 79.6 us, 288 of 48 89.6).
// At least two blocks per split, and at most 128 (head_dim 128: 64) splits, bound what the merge has to read (one
// sequence, 4096 keys: two blocks each 10.8 us, one each 13.6; head_dim 128, 2 x 4 pairs, 8192 keys: 64 splits 16.6 us,
// 128 23.7).  Returns the scratch bytes the partials need.
size_t decode_plan(const segpt_attn_params& p, int* kend_out, int* splits_out, int* chunk_out) {
  int kend = p.Sk;
  if (p.causal && p.Sq + p.q_start < kend) kend = p.Sq + p.q_start;
  constexpr int kCUs = 256;
  const int groups = (p.B * p.Hkv + 3) / 4;
  const int blocks = (kend + kDecBlock - 1) / kDecBlock;
  // (the last bound keeps the partials of many query rows within what 24576 / 8192 rows take)
  const int64_t rows = (int64_t)p.B * p.H * p.Sq, most_rows = p.D == 64 ? 24576 : 8192;
  const int most = (int)std::min<int64_t>(p.D == 64 ? kMaxSplits : kMaxSplits / 2, std::max<int64_t>(1, most_rows / rows));
  int best_per = 0;
  double best = 0;
  for (int round = 1; round <= 3; ++round) {
    int s = kCUs * round / groups;
    s = s < 1 ? 1 : (s > most ? most : s);
    int per = (blocks + s - 1) / s;
    if (per < 2) per = 2;
    const int64_t wgs = (int64_t)groups * ((blocks + per - 1) / per);
    const double load = (double)((wgs + kCUs - 1) / kCUs) * per * (1.0 + 0.03 * (round - 1));
    if (!best_per || load < best) { best = load; best_per = per; }
  }
  *kend_out = kend;
  *splits_out = (blocks + best_per - 1) / best_per;
  *chunk_out = best_per * kDecBlock;
  return (size_t)p.B * p.Hkv * *splits_out * (p.H / p.Hkv * p.Sq) * ((size_t)p.D + 2) * sizeof(float);
}

template <int D>
void launch_split(const KArgs& a, dim3 grid, hipStream_t st) {
  const bool vres = a.p.v_first.ptr != nullptr;
  if (a.p.rope_cos) {
    if (vres) hipLaunchKernelGGL((decode_split_kernel<D, true, true>), grid, dim3(kDecThreads), 0, st, a);
    else hipLaunchKernelGGL((decode_split_kernel<D, true, false>), grid, dim3(kDecThreads), 0, st, a);
  } else {
    if (vres) hipLaunchKernelGGL((decode_split_kernel<D, false, true>), grid, dim3(kDecThreads), 0, st, a);
    else hipLaunchKernelGGL((decode_split_kernel<D, false, false>), grid, dim3(kDecThreads), 0, st, a);
  }
}

int launch_fwd_decode_bf16(KArgs a, hipStream_t st) {
  const segpt_attn_params& p = a.p;
  decode_plan(p, &a.dec_kend, &a.dec_splits, &a.dec_chunk);
  char* ws = reinterpret_cast<char*>(p.kv_workspace);
  a.dec_part = reinterpret_cast<float*>(ws);
  a.dec_stat = a.dec_part + (size_t)p.B * p.H * p.Sq * a.dec_splits * p.D;
  const dim3 grid((unsigned)((p.B * p.Hkv + 3) / 4 * a.dec_splits));
  if (p.D == 64) launch_split<64>(a, grid, st);
  else if (p.D == 128) launch_split<128>(a, grid, st);
  else return (int)hipErrorInvalidValue;
  int rc = (int)hipGetLastError();
  if (rc) return rc;
  hipLaunchKernelGGL(decode_merge_kernel, dim3((unsigned)(p.B * p.Hkv * (p.H / p.Hkv) * p.Sq)), dim3(kMergeThreads), 0, st, a);
  return (int)hipGetLastError();
}

}  // namespace segpt
