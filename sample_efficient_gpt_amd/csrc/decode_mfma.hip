// bf16 forward for decode-shaped calls: a handful of query rows (H/Hkv * Sq <= 32 per kv head) against a long
// key/value cache (the reference's generation path: attention.py:191-198 builds q_start = past length,
// KVCache :15-27 grows K/V, the module masks with k_idx <= q_start + q_idx, :72-78).
//
// The training kernel would run B*H workgroups that each walk the whole cache; here the KEYS are split
// ("flash decoding"): wave (b, kv head g, split s, stream w) handles part of one chunk of the cache for ALL query
// rows of the group (n = hq * Sq + i, at most 32 = one MFMA column block), writes an unnormalised partial
// (running maximum M, sum L, O) and a second tiny kernel merges streams and splits.  Memory-bound by design: every
// K / V row is read exactly once from HBM, so the key normalisation, the rotary embedding and the value
// residual mix are done on the fly in registers (no pre-pass, no normalised copy).
//
// Per wave and 32-key block (orientation as in the training forward: lane = query column):
//   K rows from LDS in the MFMA A layout (row = key, 16-byte chunks), rotated if asked, times
//   b_j = rsqrt(mean k^2 + eps), packed to bf16                                            S^T = Khat . Qhat^T  (4 or 8 MFMAs)
//   online softmax per lane, P^T packed to bf16 = B operand
//   V rows by transposing LDS reads                                                        O^T += V'^T . P^T
#include <algorithm>

#include "mfma_common.hpp"
#include "ring_protocol.hpp"

namespace segpt {
namespace {

constexpr int kDecThreads = 256;  // 4 waves
constexpr int kDecBlock = 32;     // keys per step of a wave
constexpr int kMaxSplits = 512;
constexpr int kStreams = 4;        // a split's 32-key blocks are dealt out to four streams: blocks w, w + 4, ...
constexpr int kSplitRows = 32;     // rows of scratch per split: four streams of up to 8 query rows, or merged ones of up to 32

// LDS regions below are private to a wave: program order is enough, the compiler only has to keep it
__device__ __forceinline__ void wave_lds_sync() {
  __builtin_amdgcn_fence(__ATOMIC_ACQ_REL, "wavefront");
  __builtin_amdgcn_wave_barrier();
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
// c1 v + c2 f of eight elements, in fp32, rounded once
__device__ __forceinline__ bf16x8 mix8(bf16x8 v, bf16x8 f, float c1, float c2) {
  const u32x4 a = __builtin_bit_cast(u32x4, v), b = __builtin_bit_cast(u32x4, f);
  u32x4 w;
#pragma unroll
  for (int i = 0; i < 4; ++i) w[i] = pack_bf16x2(fmaf(c2, bf16lo(b[i]), c1 * bf16lo(a[i])), fmaf(c2, bf16hi(b[i]), c1 * bf16hi(a[i])));
  return as_bf16x8(w);
}
// (maximum, sum) of a split from those of its streams, at(w), and the streams' weights; a stream with nothing visible has
// (-inf, 0): weight 0
template <typename At>
__device__ __forceinline__ float2 merge_streams(At at, float (&w)[kStreams]) {
  float2 ml[kStreams];
#pragma unroll
  for (int i = 0; i < kStreams; ++i) ml[i] = at(i);
  const float m = fmaxf(fmaxf(ml[0].x, ml[1].x), fmaxf(ml[2].x, ml[3].x)), mu = m == -INFINITY ? 0.f : m;
#pragma unroll
  for (int i = 0; i < kStreams; ++i) w[i] = fast_exp2(ml[i].x - mu);
  return make_float2(m, (ml[0].y * w[0] + ml[1].y * w[1]) + (ml[2].y * w[2] + ml[3].y * w[3]));
}
// this wave's LDS reads have returned (before the tile they came from is requested over)
__device__ __forceinline__ void wait_lds_reads() {
  wave_lds_sync();
  __builtin_amdgcn_s_waitcnt(0xC07F);  // lgkmcnt(0) only
}

// One wave per (batch, kv head, split, stream).
// MERGED == false (at most 8 query rows per kv head: a generation step): the four waves of a workgroup take the SAME keys
// of four consecutive (batch, kv head) pairs, so that with a rotary embedding the table rows of a key block (as long as a K row
// each: cos and sin together as much as K and V) come in once per workgroup, double-buffered one block ahead.  Each wave
// writes its own partial (M, L, O) of its live query rows.
// MERGED == true (more rows, whose four partials would outgrow the scratch): the four waves take the four streams of one
// split of one pair and merge them through LDS; every lane reads its key's table rows itself.
//
// Bound by HBM: every K and V row once.  What the memory system needs for that is whole lines and requests that stay in
// flight, so K, V, V_first and the tables all travel by direct global->LDS loads into swizzled tiles (see the request
// order below).  Before, every lane loaded 16-byte pieces of its own row and, with a rotary embedding, of the two
// table rows, by each wave for itself.  Both kernels, B = 32, 18 / 6 heads, 8192 keys, head_dim 64 (403 MB): 121 -> 76.8 us
// with a rotary embedding, 83 -> 77 without; B = 8, 16 / 4 heads, 5001 keys, head_dim 128 (82 MB): 34.0 -> 22.8 us; MERGED,
// 4 x 18 / 6 heads, 4 queries, 3000 keys: 18.5 -> 16.1.
//
// The operands are rounded where the training kernels round them: keys normalised in fp32, then to bf16; probabilities
// against the exact running maximum of the wave's keys, so that the largest is 1.  Cheaper forms (the normaliser on the 16
// scores a lane holds and the raw key bits as operand; a fixed softmax reference where the QK-norm bound allows one)
// cost 3 to 5 % of accuracy (3.2e-3 -> 3.3e-3 from float64, in norm) and moved every output by 4e-3.
// A value residual is mixed in fp32 and rounded once, on the transposed fragments of V and V_first (elementwise, so the
// layout does not matter).  Two products with c1 P and c2 P are a little faster (32 x 6 pairs, 8192 keys: 110 us against 112),
// but their roundings do not cancel where the two parts do: v_first = v, coefficients (0.9, -0.85): 4e-2 from the exact mix.
// Only the block that holds the last visible key is masked, and the accumulators are rescaled only where a maximum moved.
// workgroups per CU that LDS (tiles and tables) and registers allow
template <int D, bool ROPE, bool VRES>
constexpr int kDecOcc = D == 64 ? (VRES ? 2 : 3) : (ROPE || VRES ? 1 : 2);

template <int D, bool ROPE, bool VRES, bool MERGED>
__global__ __launch_bounds__(kDecThreads, (kDecOcc<D, ROPE, VRES>)) void decode_split_kernel(KArgs a) {
  constexpr bool TABLES = ROPE && !MERGED;  // table rows staged through LDS
  constexpr int KS = D / 16;
  constexpr int MB = D / 32;
  using Z = Swz<D, kDecBlock>;
  const segpt_attn_params& p = a.p;
  __shared__ __attribute__((aligned(1024))) char tab[TABLES ? 2 * 2 * Z::kTileBytes : 16];  // [buffer][cos, sin] of a key block
  __shared__ __attribute__((aligned(1024))) char tiles[4][VRES ? 3 : 2][Z::kTileBytes];  // wave-private K, V (, V_first) rows
  __shared__ __attribute__((aligned(16))) float gsm[D];
  __shared__ float2 stat[4][MERGED ? 32 : 1];

  const int tid = threadIdx.x, lane = tid & 63;
  const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
  const int ln = lane & 31, hh = lane >> 5;
  const int rep = p.H / p.Hkv;
  const int n_rows = rep * p.Sq;  // query rows of this kv head, <= 32
  const int units = a.dec_splits * (MERGED ? 1 : kStreams), unit = blockIdx.x % units;
  const int split = MERGED ? unit : unit / kStreams, stream = MERGED ? wave : unit % kStreams;
  const int bg_all = p.B * p.Hkv, bg_raw = MERGED ? (int)(blockIdx.x / units) : 4 * (int)(blockIdx.x / units) + wave;
  // this wave's 32-key blocks: first, first + kStep, ... below k_hi; the last streams of a ragged split may have none
  constexpr int kStep = kStreams * kDecBlock;
  const int first = split * a.dec_chunk + stream * kDecBlock, k_hi = min((split + 1) * a.dec_chunk, a.dec_kend);
  const bool active = bg_raw < bg_all;  // wave-uniform; an idle wave of the last workgroup only keeps the barriers
  const int bg = active ? bg_raw : bg_all - 1;
  const int g = bg % p.Hkv, b = bg / p.Hkv;

  const int2 src = swz_src<D>(lane, wave);
  const uint32_t tab0 = lds_addr_of(tab);
  auto issue_tables = [&](int jb, int buf) {
    const int64_t row0 = (int64_t)(p.rope_k_pos0 + jb) * (D / 2);
    issue_tile_pair<D, kDecBlock>(reinterpret_cast<const char*>(p.rope_cos + row0), reinterpret_cast<const char*>(p.rope_sin + row0),
                                  tile_lane_offsets<D, kDecBlock>(D * 2, D * 2, p.Sk - jb, src.x, src.y),
                                  tab0 + buf * 2 * Z::kTileBytes + wave * 1024);
  };
  if constexpr (TABLES) { if (first < k_hi) issue_tables(first, 0); }
  // Every row travels global -> LDS as part of whole lines (a row-per-lane load covers 32 bytes of each of 32 rows and
  // leaves the rest of their lines to the L1, which 64 KB in flight overrun).  One buffer per tensor: a tile is requested
  // again as soon as its last reader has its fragments, so K is in flight during the softmax and the V product, V during
  // the next block's scores.  Order of the requests: [tables, K, V, V_first] of block 0, then tables, K, V, V_first of
  // each next block; every wait below leaves exactly the younger ones in flight.
  constexpr ring::DecodeLoads kLoads{TABLES ? 2 * Z::kPasses : 0, WaveTile<D>::kLoads, VRES ? WaveTile<D>::kLoads : 0};
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
  if (active && first < k_hi) {
    issue_k(first);
    issue_v(first);
    issue_first(first);
  }

  // ---- this lane's query (B operand column n): Qhat = sm_scale*log2e * a q g_q g_k, zero for padding columns
  if (tid < D) gsm[tid] = gprod_at(p, tid) * p.sm_scale * kLog2e;
  __syncthreads();
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
  float m_run = -INFINITY, l_run[2] = {0.f, 0.f};  // l_run: this lane's half of the keys, as two partial sums

  const uint32_t row16 = tab0 + swz_off_row16<D>(lane);
  const uint32_t krm = ktile + swz_off_rm<D>(lane), vtr = vtile + swz_off_tr<D>(lane), ftr = ftile + swz_off_tr<D>(lane);
  int buf = 0;
  wait_vmcnt<0>();  // nothing but tile requests may be in flight in the loop, whose waits count them
  wave_lds_sync();
  for (int jb = first; jb < k_hi; jb += kStep) {
    const bool more = jb + kStep < k_hi;
    if (active) wait_vmcnt<ring::decode_kept_at_top(kLoads)>();  // this block's tables and K
    else wait_vmcnt<0>();
    if constexpr (TABLES) {
      __syncthreads();  // every wave's pieces of the tables are there, and nobody reads the other buffer any more
      if (more) issue_tables(jb + kStep, buf ^ 1);
    }
    if (active) {
      wave_lds_sync();
      u32x4 kraw[KS];
#pragma unroll
      for (int ks = 0; ks < KS; ++ks) kraw[ks] = __builtin_bit_cast(u32x4, swz_frag_rm<D>(krm, 0, ks));
      wait_lds_reads();
      if (more) issue_k(jb + kStep);
      float x[KS][8];
      unpack_b_layout<KS>(kraw, x);
      if constexpr (ROPE && MERGED) {
        const int64_t pos = (int64_t)(p.rope_k_pos0 + min(jb + ln, p.Sk - 1)) * (D / 2);
        rope_b_layout<KS>(x, p.rope_cos + pos, p.rope_sin + pos, hh);
      } else if constexpr (ROPE) {
        const uint32_t cos16 = row16 + buf * 2 * Z::kTileBytes, sin16 = cos16 + Z::kTileBytes;
#pragma unroll
        for (int ks = 0; ks < KS / 2; ++ks)
#pragma unroll
          for (int i = 0; i < 2; ++i) {
            const uint32_t off = (uint32_t)((4 * ks + 2 * hh + i) << 4);  // floats 16 ks + 8 hh + 4 i ..
            const f32x4 c = lds_read_f4(cos16 ^ off), sn = lds_read_f4(sin16 ^ off);
#pragma unroll
            for (int t = 0; t < 4; ++t) rope_pair(x[ks][4 * i + t], x[ks + KS / 2][4 * i + t], c[t], sn[t]);
          }
      }
      float ss = 0.f;
#pragma unroll
      for (int ks = 0; ks < KS; ++ks)
#pragma unroll
        for (int t = 0; t < 8; ++t) ss += x[ks][t] * x[ks][t];
      ss = half_sum(ss);
      const float beta = row_normaliser_fast(p, ss, 1.0f / D);
      f32x16 s = splat16(0.f);
#pragma unroll
      for (int ks = 0; ks < KS; ++ks) {
        u32x4 w;
#pragma unroll
        for (int i = 0; i < 4; ++i) w[i] = pack_bf16x2(x[ks][2 * i] * beta, x[ks][2 * i + 1] * beta);
        s = mfma32(as_bf16x8(w), qreg[ks], s);
      }
      // register r holds key jb + 4hh + c_r, c_r = 8(r/4) + r%4
      if (jb + kDecBlock - 1 > min(all_see, k_hi - 1)) {  // visible iff <= qlim and < k_hi
        const int t = min(qlim, k_hi - 1) - jb - 4 * hh;
#pragma unroll
        for (int r = 0; r < 16; ++r)
          if (8 * (r >> 2) + (r & 3) > t) s[r] = -INFINITY;
      }
      float mx = s[0];
#pragma unroll
      for (int r = 1; r < 16; ++r) mx = fmaxf(mx, s[r]);
      mx = half_max(mx);
      const float m_new = fmaxf(m_run, mx);
      const float mu = m_new == -INFINITY ? 0.f : m_new;  // nothing visible yet: keep exp2 away from inf - inf
      if (__builtin_amdgcn_ballot_w64(mx > m_run) != 0) {  // elsewhere the factor is 1
        const float corr = fast_exp2(m_run - mu);  // m_run = -inf gives 0
        l_run[0] *= corr;
        l_run[1] *= corr;
#pragma unroll
        for (int mb = 0; mb < MB; ++mb)
#pragma unroll
          for (int r = 0; r < 16; ++r) oacc[mb][r] *= corr;
      }
      m_run = m_new;
#pragma unroll
      for (int r = 0; r < 16; ++r) s[r] = fast_exp2(s[r] - mu);
      if (more) wait_vmcnt<ring::decode_kept_before_v(kLoads, true)>(); else wait_vmcnt<ring::decode_kept_before_v(kLoads, false)>();  // this block's V (and V_first)
      const bf16x8 pb[2] = {pack_c_half_sum(s, 0, l_run), pack_c_half_sum(s, 1, l_run)};
      wave_lds_sync();
#pragma unroll
      for (int mb = 0; mb < MB; ++mb)
#pragma unroll
        for (int s2 = 0; s2 < 2; ++s2) {
          bf16x8 vT = swz_frag_tr<D>(vtr, mb, s2);
          if constexpr (VRES) vT = mix8(vT, swz_frag_tr<D>(ftr, mb, s2), c1, c2);
          oacc[mb] = mfma32(vT, pb[s2], oacc[mb]);
        }
      wait_lds_reads();
      if (more) {
        issue_v(jb + kStep);
        issue_first(jb + kStep);
      }
    }
    buf ^= 1;
  }

  const float l_tot = half_sum(l_run[0] + l_run[1]);
  if constexpr (MERGED) {
    // ---- merge the four streams (different keys, same queries): partial rows n of [bg, split][n_rows][D]
    float (*osm)[D][32] = reinterpret_cast<float (*)[D][32]>(tiles[0][0]);
    static_assert(sizeof(tiles) >= 4 * D * 32 * sizeof(float), "the tiles' memory holds the four accumulators");
    __syncthreads();  // every wave is done with its tiles
    if (hh == 0) stat[wave][ln] = make_float2(m_run, l_tot);
#pragma unroll
    for (int mb = 0; mb < MB; ++mb)
#pragma unroll
      for (int r = 0; r < 16; ++r) osm[wave][32 * mb + 8 * (r >> 2) + 4 * hh + (r & 3)][ln] = oacc[mb][r];
    __syncthreads();
    const int64_t at = ((int64_t)bg * units + unit) * n_rows;
    for (int e = tid; e < 32 * D; e += kDecThreads) {
      const int n = e % 32, d = e / 32;
      if (n >= n_rows) continue;
      float w[kStreams];
      const float2 ml = merge_streams([&](int i) { return stat[i][n]; }, w);
      a.dec_part[(at + n) * D + d] = (osm[0][d][n] * w[0] + osm[1][d][n] * w[1]) + (osm[2][d][n] * w[2] + osm[3][d][n] * w[3]);
      if (d == 0) *reinterpret_cast<float2*>(a.dec_stat + (at + n) * 2) = ml;
    }
  } else if (active && qlive) {
    // ---- this wave's partial: rows n of [bg, unit][n_rows][D]
    const int64_t at = ((int64_t)bg * units + unit) * n_rows + ln;
#pragma unroll
    for (int mb = 0; mb < MB; ++mb)
#pragma unroll
      for (int q = 0; q < 4; ++q)
        *reinterpret_cast<float4*>(a.dec_part + at * D + 32 * mb + 8 * q + 4 * hh) =
            make_float4(oacc[mb][4 * q], oacc[mb][4 * q + 1], oacc[mb][4 * q + 2], oacc[mb][4 * q + 3]);
    if (hh == 0) *reinterpret_cast<float2*>(a.dec_stat + at * 2) = make_float2(m_run, l_tot);
  }
}

// One workgroup per (batch, kv head, query row): merges the streams of each split, then the splits, normalises, gates,
// writes y (bf16) and lse (natural log).  Thread (group gi, column d) sums the splits gi, gi + G, ... of output column d
// (G = threads / D); its first partial values are requested before the statistics are reduced, so that the kernel is
// about two memory round trips long whatever the number of splits.  Every sum has a fixed order: deterministic.
constexpr int kMergeThreads = 256;
constexpr int kMergeEarly = 16;  // partial values per thread requested up front

template <int W>  // partials per split
__global__ __launch_bounds__(kMergeThreads) void decode_merge_kernel(KArgs a) {
  const segpt_attn_params& p = a.p;
  constexpr int kEarly = kMergeEarly / W;
  __shared__ float wsm[kMaxSplits];         // weight of a split
  __shared__ float wst[W][kMaxSplits];      // weight of a stream within its split
  __shared__ float redm[4], redl[4];
  __shared__ float part[kMergeThreads];
  const int D = p.D, tid = threadIdx.x, lane = tid & 63, wave = tid >> 6;
  const int rep = p.H / p.Hkv;
  const int n_rows = rep * p.Sq;
  const int n = blockIdx.x % n_rows, bg = blockIdx.x / n_rows;
  const int g = bg % p.Hkv, b = bg / p.Hkv;
  const int S = a.dec_splits;
  const int G = kMergeThreads / D, gi = tid / D, d = tid - gi * D;
  const float* col = a.dec_part + ((int64_t)bg * S * W * n_rows + n) * D + d;  // stream w of split sp: + (sp * W + w) * part_step
  const float2* stat = reinterpret_cast<const float2*>(a.dec_stat) + (int64_t)bg * S * W * n_rows + n;
  const int64_t part_step = (int64_t)n_rows * D;
  float pv[kEarly][W];
#pragma unroll
  for (int u = 0; u < kEarly; ++u)
#pragma unroll
    for (int w = 0; w < W; ++w) {
      const int sp = gi + G * u;
      pv[u][w] = sp < S ? col[(sp * W + w) * part_step] : 0.f;
    }
  auto split_stat = [&](int sp, float (&ws)[W]) {
    if constexpr (W == 1) {
      ws[0] = 1.f;
      return stat[sp * n_rows];
    } else {
      return merge_streams([&](int w) { return stat[(sp * W + w) * n_rows]; }, ws);
    }
  };
  float m = -INFINITY, ws[W];
  for (int sp = tid; sp < S; sp += kMergeThreads) m = fmaxf(m, split_stat(sp, ws).x);
#pragma unroll
  for (int o = 1; o < 64; o <<= 1) m = fmaxf(m, __shfl_xor(m, o, 64));
  if (lane == 0) redm[wave] = m;
  __syncthreads();
  const float M = fmaxf(fmaxf(redm[0], redm[1]), fmaxf(redm[2], redm[3]));
  float l = 0.f;
  for (int sp = tid; sp < S; sp += kMergeThreads) {
    const float2 ml = split_stat(sp, ws);
    const float w = exp2f(ml.x - M);
    wsm[sp] = w;
#pragma unroll
    for (int i = 0; i < W; ++i) wst[i][sp] = ws[i];
    l += ml.y * w;
  }
#pragma unroll
  for (int o = 1; o < 64; o <<= 1) l += __shfl_xor(l, o, 64);
  if (lane == 0) redl[wave] = l;
  __syncthreads();  // also publishes the weights
  const float L = (redl[0] + redl[1]) + (redl[2] + redl[3]);
  float acc = 0.f;
  auto add_split = [&](int sp, const float (&o)[W]) {
    if constexpr (W == 1) acc += o[0] * wsm[sp];
    else acc += ((o[0] * wst[0][sp] + o[1] * wst[1][sp]) + (o[2] * wst[2][sp] + o[3] * wst[3][sp])) * wsm[sp];
  };
#pragma unroll
  for (int u = 0; u < kEarly; ++u) {
    const int sp = gi + G * u;
    if (sp < S) add_split(sp, pv[u]);
  }
#pragma unroll 4
  for (int sp = gi + G * kEarly; sp < S; sp += G) {
    float o[W];
#pragma unroll
    for (int w = 0; w < W; ++w) o[w] = col[(sp * W + w) * part_step];
    add_split(sp, o);
  }
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

bool merged_streams(const segpt_attn_params& p) { return p.H / p.Hkv * p.Sq * kStreams > kSplitRows; }

// Split plan of a decode-shaped call: keys [0, kend) in `splits` chunks of `chunk` keys (a multiple of 128, no empty
// split), enough for one resident round of the card: 768 (batch, kv head, split) at head_dim 64, 256 at 128.  What a
// workgroup takes (see the kernel) does not change the plan, which fixes the reference every probability is rounded
// against, nor the number of workgroups.  Returns the scratch bytes the partials need, at most 32 rows per (pair, split).
size_t decode_plan(const segpt_attn_params& p, int* kend_out, int* splits_out, int* chunk_out) {
  int kend = p.Sk;
  if (p.causal && p.Sq + p.q_start < kend) kend = p.Sq + p.q_start;
  constexpr int kSplitKeys = kStreams * kDecBlock;
  const int pairs = p.B * p.Hkv;
  int s = ((p.D == 64 ? 768 : 256) + pairs - 1) / pairs;
  s = std::max(1, std::min({s, (kend + kSplitKeys - 1) / kSplitKeys, kMaxSplits}));
  const int per = (kend + s - 1) / s;
  const int chunk = std::max(1, (per + kSplitKeys - 1) / kSplitKeys) * kSplitKeys;
  s = (kend + chunk - 1) / chunk;
  *kend_out = kend; *splits_out = s; *chunk_out = chunk;
  return (size_t)pairs * s * (merged_streams(p) ? 1 : kStreams) * (p.H / p.Hkv * p.Sq) * ((size_t)p.D + 2) * sizeof(float);
}

template <int D, bool MERGED>
void launch_split(const KArgs& a, hipStream_t st) {
  const segpt_attn_params& p = a.p;
  const dim3 grid((unsigned)(MERGED ? p.B * p.Hkv * a.dec_splits : (p.B * p.Hkv + 3) / 4 * a.dec_splits * kStreams)), block(kDecThreads);
  const bool vres = p.v_first.ptr != nullptr;
  if (p.rope_cos) {
    if (vres) hipLaunchKernelGGL((decode_split_kernel<D, true, true, MERGED>), grid, block, 0, st, a);
    else hipLaunchKernelGGL((decode_split_kernel<D, true, false, MERGED>), grid, block, 0, st, a);
  } else {
    if (vres) hipLaunchKernelGGL((decode_split_kernel<D, false, true, MERGED>), grid, block, 0, st, a);
    else hipLaunchKernelGGL((decode_split_kernel<D, false, false, MERGED>), grid, block, 0, st, a);
  }
}

int launch_fwd_decode_bf16(KArgs a, hipStream_t st) {
  const segpt_attn_params& p = a.p;
  decode_plan(p, &a.dec_kend, &a.dec_splits, &a.dec_chunk);
  const bool merged = merged_streams(p);
  char* ws = reinterpret_cast<char*>(p.kv_workspace);
  a.dec_part = reinterpret_cast<float*>(ws);
  a.dec_stat = a.dec_part + (size_t)p.B * p.H * p.Sq * a.dec_splits * (merged ? 1 : kStreams) * p.D;
  if (p.D == 64) merged ? launch_split<64, true>(a, st) : launch_split<64, false>(a, st);
  else if (p.D == 128) merged ? launch_split<128, true>(a, st) : launch_split<128, false>(a, st);
  else return (int)hipErrorInvalidValue;
  int rc = (int)hipGetLastError();
  if (rc) return rc;
  const dim3 rows((unsigned)(p.B * p.Hkv * (p.H / p.Hkv) * p.Sq));
  if (merged) hipLaunchKernelGGL(decode_merge_kernel<1>, rows, dim3(kMergeThreads), 0, st, a);
  else hipLaunchKernelGGL(decode_merge_kernel<kStreams>, rows, dim3(kMergeThreads), 0, st, a);
  return (int)hipGetLastError();
}

}  // namespace segpt
