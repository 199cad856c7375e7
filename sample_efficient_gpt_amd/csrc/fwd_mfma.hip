// bf16 forward: causal GQA flash attention on the normalised keys of the key/value pre-pass.
//
// Workgroup = 4 waves (two or three workgroups share a CU at head_dim 64 so that one's softmax overlaps the
// others' MFMAs); wave w owns NQB blocks of 32 queries (see FwdShape).  Scores are produced TRANSPOSED,
//   S^T[key][query] = Khat[key][:] . Qhat[query][:]          (A = Khat tile from LDS, B = Qhat registers)
// so every lane owns one query column: the softmax state (reference point, row sum) is a per-lane scalar,
// row reductions are in-register plus one exchange with lane^32, and the bf16 probabilities are already
// laid out as the B operand of
//   O^T[d][query] += V'^T[d][key] . P^T[key][query]          (A = transposing LDS read of the V' tile).
// Qhat = sm_scale*log2(e) * a_i * q_i * g_q * g_k  (both scale vectors live on the query side) is formed in
// the prologue; Khat = b_j * k_j and V' = c1 v + c2 v_first are read as written by the pre-pass.
#include <algorithm>

#include "mfma_common.hpp"
#include "ring_protocol.hpp"

namespace segpt {
namespace {

// Khat / V' come from the key/value pre-pass (bf16, contiguous [B,Hkv,Sk,D]) and travel global->LDS
// directly into a swizzled ring of stages, so the loop holds no staging registers and no normalisation
// work.  Software pipeline over 32-key blocks n (two per staged tile), one barrier per tile:
//   B(n)   S^T MFMAs from the row-major Khat fragments requested one block earlier
//   C(n)   request the transposed V' fragments of block n
//   D(n)   mask (diagonal blocks only), exp2, bf16 pack, row sums
//   A(n+1) request the row-major Khat fragments of block n+1 (possibly of the next tile, already landed)
//   E(n)   O^T += V'^T P^T MFMAs
// Two shapes at head_dim 64.  WIDE: 64 query rows per wave (K fragments shared by two query blocks), four LDS
// stages, two workgroups per CU: best when a workgroup streams many key tiles (S = 8192: 7 % faster than
// NARROW).  NARROW: 32 rows per wave, three stages (48 KB), three workgroups per CU: twice as many, lighter
// workgroups whose start-up / write-out latencies hide behind two neighbours instead of one (S = 2048: 1 %
// faster, S = 1152: 10 %, S = 768: 13 %, S = 384: 27 %).  The launcher picks by the number of keys.
// head_dim 128: 32 rows per wave and 32-KEY tiles (a tile pair is then the same 16 KB as at head_dim 64, a block of a
// tile carries twice the MFMAs, so one block per tile keeps the ratio of barriers and tile loads to MFMAs), four stages
// = 64 KB, two workgroups per CU.  With 64-key tiles the ring alone is 96 KB and a CU holds one workgroup, i.e. one
// wave per SIMD with nothing to overlap its softmax phase with.
// PARTS == 2 (see fwd_parts()): the workgroup owns 64 query rows, two waves each take one of the two 32-key blocks of
// every 64-key tile for the same rows, and the pair merges its softmax states through LDS behind the loop.
template <int D, bool WIDE, int PARTS = 1>
struct FwdShape {
  static constexpr int kNQB = (D == 64 && WIDE && PARTS == 1) ? 2 : 1;  // 32-query blocks per wave
  static constexpr int kBK = D == 64 || PARTS == 2 ? 64 : 32;           // keys per streamed tile
  static constexpr int kStages = PARTS == 2 ? 3 : (D == 64 ? (WIDE ? 4 : 3) : 4);
  static constexpr int kOcc = PARTS == 2 ? (D == 64 ? 3 : 1) : (D == 64 ? (WIDE ? 2 : 3) : 2);
  static constexpr int kRowWaves = 4 / PARTS;             // waves side by side along the query rows
  static constexpr int kBQ = kRowWaves * 32 * kNQB;
  static constexpr int kStoreUnits = D / 64;              // partial results of a split launch, in 32 KB
};

// ROPE (rope tables given) is a compile-time switch so that the table rows are ordinary, unconditional loads that
// travel with the start-up tiles instead of costing a memory round trip of their own behind a branch.
//
// SPLIT: workgroup (tile, head, batch; y = share s) takes only the key tiles [s, s + 1) * fwd_chunk of its query tile
// and, unless that is all of them, leaves an unnormalised partial (reference m, sum l, O in fp32) for
// fwd_merge_kernel; see fwd_split_plan() for when.
template <int D, bool WIDE, bool ROPE, bool SPLIT, int PARTS>
__global__ __launch_bounds__(kThreadsM, (FwdShape<D, WIDE, PARTS>::kOcc)) void fwd_bf16_kernel(KArgs a) {
  using F = FwdShape<D, WIDE, PARTS>;
  static_assert(PARTS == 1 || (PARTS == 2 && !SPLIT && F::kNQB == 1 && F::kBK == 64), "a tile has two 32-key blocks");
  constexpr bool kMayMissKeys = SPLIT || PARTS == 2;  // a row may have no visible key among those a wave sees
  constexpr int NQB = F::kNQB, BQ = F::kBQ, NS = F::kStages, BK = F::kBK;
  constexpr int kBlocksPerTile = BK / 32;
  using Z = Swz<D, BK>;
  constexpr int KS = D / 16;
  constexpr int MB = D / 32;
  constexpr int kStageBytes = 2 * Z::kTileBytes;
  constexpr int kLoadsPerTile = 2 * Z::kPasses;  // per wave
  const segpt_attn_params& p = a.p;
  __shared__ __attribute__((aligned(1024))) char lds[NS * kStageBytes];
  __shared__ __attribute__((aligned(16))) float gsm[D];  // sm_scale*log2e * g_q * g_k, read as float4 slices

  const int tid = threadIdx.x, lane = tid & 63;
  const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);  // wave-uniform: everything derived from it stays scalar
  const int ln = lane & 31, hh = lane >> 5;
  const int rep = p.H / p.Hkv;
  const int n_qt = (p.Sq + BQ - 1) / BQ;
  const WgCoord wg = decode_wg(!SPLIT && F::kOcc >= 2 ? balanced_id(blockIdx.x, gridDim.x) : (int)blockIdx.x, n_qt, p.B, p.Hkv, rep, wg_pinned_pairs(p.B, p.Hkv, false));
  if (!wg.valid) return;  // idle padding workgroup (whole workgroup, before any barrier)
  const int b = wg.b, g = wg.g, h = wg.g * rep + wg.hh;
  const int q0 = wg.tile * BQ;
  const int row_wave = PARTS == 1 ? wave : wave % F::kRowWaves, part = PARTS == 1 ? 0 : wave / F::kRowWaves;
  const int qw0 = q0 + row_wave * 32 * NQB;  // first query of this wave

  int kend = p.Sk;
  if (p.causal) kend = min(p.Sk, q0 + BQ + p.q_start);
  const int all_kt = (kend + BK - 1) / BK;
  // this workgroup's keys: k0 .. kend - 1; everything below counts keys from k0
  const int share = SPLIT ? (int)blockIdx.y : 0, k0 = SPLIT ? share * a.fwd_chunk * BK : 0;
  if (SPLIT && k0 >= kend) return;
  const int Sk = p.Sk - k0, q_start = p.q_start - k0;
  kend = SPLIT ? min(kend - k0, a.fwd_chunk * BK) : kend;
  const int n_kt = (kend + BK - 1) / BK;
  const char* kbase = reinterpret_cast<const char*>(a.khat + (((int64_t)b * p.Hkv + g) * p.Sk + k0) * D);
  const char* vbase = a.vmix ? reinterpret_cast<const char*>(a.vmix + (((int64_t)b * p.Hkv + g) * p.Sk + k0) * D)
                             : reinterpret_cast<const char*>(row_ptr<uint16_t>(p.v, b, g, k0));
  const uint32_t kstep = D * 2, vstep = a.vmix ? (uint32_t)D * 2 : (uint32_t)p.v.stride_s * 2;

  const uint32_t lds0 = lds_addr_of(lds);
  const int2 src = swz_src<D>(lane, wave);
  const uint32_t wave_dst = lds0 + wave * 1024;
  const TileLaneOff<D, BK> full_tile = tile_lane_offsets<D, BK>(kstep, vstep, BK, src.x, src.y);
  auto issue_tile = [&](int jt) {  // tile jt -> stage jt % NS
    const char* ksrc = kbase + (int64_t)jt * BK * kstep;
    const char* vsrc = vbase + (int64_t)jt * BK * vstep;
    const uint32_t dst = wave_dst + (jt % NS) * kStageBytes;
    const int left = Sk - jt * BK;
    if (left >= BK) issue_tile_pair<D, BK>(ksrc, vsrc, full_tile, dst);
    else issue_tile_pair<D, BK>(ksrc, vsrc, tile_lane_offsets<D, BK>(kstep, vstep, left, src.x, src.y), dst);
  };

  // ---- start-up.  The workgroup's query rows come in as tiles too (read row-per-lane from global memory, every
  // wave-wide load would touch 32 cache lines for 32 bytes each; staged through LDS by direct loads they are
  // whole lines, and the row-major fragment read of a tile is exactly the B-operand layout): they take the last
  // kQStages stages of the ring, the first kEarlyTiles key tiles (those that fit before them) are requested at the
  // same time, the scale vector behind them: one memory round trip.  The remaining start-up tiles follow once the
  // query rows sit in registers (run() below).
  constexpr int kQStages = (BQ + 2 * BK - 1) / (2 * BK);  // a stage holds two tiles of BK rows
  constexpr ring::Protocol R = PARTS == 1 ? ring::forward(NS, kQStages, Z::kPasses) : ring::forward_parts(NS, kQStages, Z::kPasses);  // the pipeline's numbers: ring_protocol.hpp
  static_assert(ring::well_formed(R) && R.loads_per_tile == kLoadsPerTile && !R.wait_before_loop && R.issue_at_top, "tile pipeline");
  static_assert(R.early_tiles >= ring::kTilesNeededAtLoopStart, "the loop is entered without a further wait");
#pragma unroll
  for (int t = 0; t < R.early_tiles; ++t)
    if (t < n_kt) issue_tile(t);
  {
    const char* qb = reinterpret_cast<const char*>(row_ptr<uint16_t>(p.q, b, h, q0));
#pragma unroll
    for (int i = 0; i < kQStages; ++i)
      issue_tile_pair<D, BK>(qb, qb, rowblock_lane_offsets<D, BK>((uint32_t)p.q.stride_s * 2, 2 * BK * i, min(p.Sq - q0, BQ), src.x, src.y),
                         wave_dst + (R.row_stage_first + i) * kStageBytes);
  }

  // ---- Qhat registers: B operands of S^T, [nb][ks]
  RopeB<KS> rope_b[NQB];
  if (ROPE) {
#pragma unroll
    for (int nb = 0; nb < NQB; ++nb) {
      const int64_t pos = (int64_t)(p.rope_q_pos0 + min(qw0 + 32 * nb + ln, p.Sq - 1)) * (D / 2);
      rope_b[nb] = rope_b_load<KS>(p.rope_cos + pos, p.rope_sin + pos, hh);
    }
  }
  float gval = 0.f;
  if (tid < D) gval = gprod_at(p, tid) * p.sm_scale * kLog2e;
  if (tid < D) gsm[tid] = gval;
  wait_vmcnt<0>();
  __syncthreads();
  const bool bounded = !(p.flags & (SEGPT_FLAG_RUNNING_MAX | SEGPT_FLAG_NO_NORM)) && logit_bound<D>(gsm, lane) <= kNoMaxBound;  // wave-uniform
  bf16x8 qreg[NQB][KS];
#pragma unroll
  for (int nb = 0; nb < NQB; ++nb) {
    const int row = min(qw0 + 32 * nb + ln, p.Sq - 1);
    // rows 32*(NQB*row_wave + nb) .. +31 of the block: which BK-row tile of the staged block, and which 32-row block of it
    const int blk = NQB * row_wave + nb, tile = blk / kBlocksPerTile, rb = blk % kBlocksPerTile;
    const uint32_t rm = lds0 + (R.row_stage_first + (tile >> 1)) * kStageBytes + (tile & 1) * Z::kTileBytes + swz_off_rm<D>(lane);
    u32x4 raw[KS];
#pragma unroll
    for (int ks = 0; ks < KS; ++ks) raw[ks] = __builtin_bit_cast(u32x4, swz_frag_rm<D>(rm, rb, ks));
    float x[KS][8];
    unpack_b_layout<KS>(raw, x);
    if (ROPE) rope_b_apply<KS>(x, rope_b[nb]);
    float ss = 0.f;
#pragma unroll
    for (int ks = 0; ks < KS; ++ks)
#pragma unroll
      for (int t = 0; t < 8; ++t) ss += x[ks][t] * x[ks][t];
    ss = half_sum(ss);
    const float alpha = row_normaliser_fast(p, ss, 1.0f / D);
#pragma unroll
    for (int ks = 0; ks < KS; ++ks) {
      const float4 ga = *reinterpret_cast<const float4*>(gsm + 16 * ks + 8 * hh);
      const float4 gb = *reinterpret_cast<const float4*>(gsm + 16 * ks + 8 * hh + 4);
      u32x4 w;
      w[0] = pack_bf16x2(x[ks][0] * alpha * ga.x, x[ks][1] * alpha * ga.y);
      w[1] = pack_bf16x2(x[ks][2] * alpha * ga.z, x[ks][3] * alpha * ga.w);
      w[2] = pack_bf16x2(x[ks][4] * alpha * gb.x, x[ks][5] * alpha * gb.y);
      w[3] = pack_bf16x2(x[ks][6] * alpha * gb.z, x[ks][7] * alpha * gb.w);
      qreg[nb][ks] = as_bf16x8(w);
    }
  }

  f32x16 oacc[MB][NQB];
#pragma unroll
  for (int mb = 0; mb < MB; ++mb)
#pragma unroll
    for (int nb = 0; nb < NQB; ++nb) oacc[mb][nb] = splat16(0.f);
  // m_ref: the value subtracted from the logits before exp2 (0 on the bounded path); l_run: this lane's
  // share of the row sum (its half of the keys; halves are added in the epilogue)
  float m_ref[NQB], l_run[NQB][2];
  int qlim[NQB];  // last visible key of this lane's query in block nb
#pragma unroll
  for (int nb = 0; nb < NQB; ++nb) {
    m_ref[nb] = bounded ? 0.f : -INFINITY;
    l_run[nb][0] = l_run[nb][1] = 0.f;
    qlim[nb] = p.causal ? min(qw0 + 32 * nb + ln + q_start, Sk - 1) : Sk - 1;
  }

  // 32-key blocks this wave has to visit (causal: up to the block holding its last query's diagonal)
  int n_act = (kend + 31) / 32;
  if (p.causal) n_act = min(n_act, (qw0 + 32 * NQB - 1 + q_start) / 32 + 1);
  if (SPLIT && p.causal && qw0 + 32 * NQB - 1 + q_start < 0) n_act = 0;

  // PARTS == 2: this wave's block of every tile is number `part` (a multiple of 4 KB further: the XOR terms stay below)
  const uint32_t rm_lane = lds0 + swz_off_rm<D>(lane) + part * 32 * Z::kRB;
  const uint32_t tr_lane = lds0 + swz_off_tr<D>(lane) + part * 32 * Z::kRB + Z::kTileBytes;  // V' tile of a stage
  bf16x8 kf[KS];
  auto request_rowmajor = [&](uint32_t rm, int kb) {  // kb compile-time at every call site
#pragma unroll
    for (int ks = 0; ks < KS; ++ks) kf[ks] = swz_frag_rm<D>(rm, kb, ks);
  };
  // One 32-key block.  MASKED / BOUNDED are compile-time so that a whole block is one straight-line
  // scheduling region (a branch in the middle would keep the compiler from interleaving the exp2 work with
  // the neighbouring MFMAs and LDS reads).
  auto step = [&](auto masked_c, auto bounded_c, uint32_t tr, int kb, int jb, uint32_t next_rm, int next_kb) {
    constexpr bool MASKED = decltype(masked_c)::value != 0, BOUNDED = decltype(bounded_c)::value != 0;
    f32x16 s[NQB];
#pragma unroll
    for (int nb = 0; nb < NQB; ++nb) s[nb] = splat16(0.f);
    // one query block's chain after the other (not interleaved): the first block's scores are complete while
    // the second block's MFMAs still run, so its exp2 work has something to hide behind
#pragma unroll
    for (int nb = 0; nb < NQB; ++nb)
#pragma unroll
      for (int ks = 0; ks < KS; ++ks) s[nb] = mfma32(kf[ks], qreg[nb][ks], s[nb]);
    bf16x8 vT[MB][2];
#pragma unroll
    for (int mb = 0; mb < MB; ++mb) {
      vT[mb][0] = swz_frag_tr<D>(tr, mb, 2 * kb);
      vT[mb][1] = swz_frag_tr<D>(tr, mb, 2 * kb + 1);
    }
    if (MASKED) {  // block touches the diagonal or the end of the keys
#pragma unroll
      for (int nb = 0; nb < NQB; ++nb) {
        // register r holds key jb + 4hh + c_r, c_r = 8(r/4) + r%4: masked iff c_r > qlim - jb - 4hh
        const int t = qlim[nb] - jb - 4 * hh;
#pragma unroll
        for (int r = 0; r < 16; ++r)
          if (8 * (r >> 2) + (r & 3) > t) s[nb][r] = -INFINITY;
      }
    }
    if (!BOUNDED) {
      // general path: lazily maintained reference, raised only when a row exceeds it by 2^kLazyThresh
#pragma unroll
      for (int nb = 0; nb < NQB; ++nb) {
        float mx = s[nb][0];
#pragma unroll
        for (int r = 1; r < 16; ++r) mx = fmaxf(mx, s[nb][r]);
        mx = half_max(mx);
        const bool need = mx > m_ref[nb] + kLazyThresh;
        if (__builtin_amdgcn_ballot_w64(need) != 0) {
          const float m_new = need ? mx : m_ref[nb];
          const float corr = kMayMissKeys && !need ? 1.f : fast_exp2(m_ref[nb] - m_new);
          m_ref[nb] = m_new;
          l_run[nb][0] *= corr;
          l_run[nb][1] *= corr;
#pragma unroll
          for (int mb = 0; mb < MB; ++mb)
#pragma unroll
            for (int r = 0; r < 16; ++r) oacc[mb][nb][r] *= corr;
        }
        const float mu = kMayMissKeys && m_ref[nb] == -INFINITY ? 0.f : m_ref[nb];
#pragma unroll
        for (int r = 0; r < 16; ++r) s[nb][r] -= mu;
      }
    }
    bf16x8 pb[2][NQB];
#pragma unroll
    for (int nb = 0; nb < NQB; ++nb) {
#pragma unroll
      for (int r = 0; r < 16; ++r) s[nb][r] = fast_exp2(s[nb][r]);
      pb[0][nb] = pack_c_half_sum(s[nb], 0, l_run[nb]);
      pb[1][nb] = pack_c_half_sum(s[nb], 1, l_run[nb]);
    }
    request_rowmajor(next_rm, next_kb);  // unconditional: past the last block the fragments are simply unused
#pragma unroll
    for (int nb = 0; nb < NQB; ++nb)
#pragma unroll
      for (int s2 = 0; s2 < 2; ++s2)
#pragma unroll
        for (int mb = 0; mb < MB; ++mb) oacc[mb][nb] = mfma32(vT[mb][s2], pb[s2][nb], oacc[mb][nb]);
  };

  // leading blocks of this wave that need no mask: every key of the block is visible to every query of the
  // wave and lies inside the key range
  int n_full = Sk / 32;
  if (p.causal) n_full = min(n_full, (qw0 + q_start + 1) / 32);
  if (SPLIT) n_full = max(0, min(n_full, kend / 32));

  // ---- pipeline.  The tile loads that stay in flight across iterations must be the youngest vector-memory
  // operations of the wave (waits are in-order): the prologue's wait left nothing else behind.
  // Protocol: at the top of iteration jt tiles jt and jt+1 have landed and tiles jt+2 .. jt+NS-2 are in
  // flight; the stage of tile jt-1 is free (everyone passed the barrier that ended iteration jt-1), so tile
  // jt+NS-1 is requested right away and has a whole iteration to land; the wait at the bottom leaves the
  // youngest NS-3 tiles in flight, i.e. tile jt+2 is complete before the barrier.
  auto run = [&](auto bounded_c) {
    __syncthreads();  // every wave has its query rows in registers: their stages are free
#pragma unroll
    for (int t = R.early_tiles; t < R.startup_tiles; ++t)
      if (t < n_kt) issue_tile(t);
    if (n_act > 0) request_rowmajor(rm_lane, 0);
    int stage = 0;
    // Two loops instead of a per-block choice inside one: each body is then a single straight-line region
    // with one variant of the block (a join of the two variants costs a copy of every accumulator).
    // Loop A: tiles whose two blocks need no mask.  Loop B: the rest (masking a fully visible block is a no-op).
    const int n_a = PARTS == 1 ? n_full / kBlocksPerTile : (n_full + 1 - part) / 2;  // n_full <= n_act, so these tiles are all active
    int jt = 0;
    for (; jt < n_a; ++jt) {
      const int nstage = stage == NS - 1 ? 0 : stage + 1;
      const bool issued = jt + R.issue_ahead < n_kt;
      if (issued) issue_tile(jt + R.issue_ahead);
      const uint32_t rm = rm_lane + stage * kStageBytes, tr = tr_lane + stage * kStageBytes;
      if constexpr (PARTS == 2) {
        step(IC<0>{}, bounded_c, tr, 0, BK * jt + 32 * part, rm_lane + nstage * kStageBytes, 0);
      } else if constexpr (kBlocksPerTile == 2) {
        step(IC<0>{}, bounded_c, tr, 0, BK * jt, rm, 1);
        step(IC<0>{}, bounded_c, tr, 1, BK * jt + 32, rm_lane + nstage * kStageBytes, 0);
      } else {
        step(IC<0>{}, bounded_c, tr, 0, BK * jt, rm_lane + nstage * kStageBytes, 0);
      }
      if (issued) wait_vmcnt<ring::loads_kept_after_iteration(R, true)>(); else wait_vmcnt<ring::loads_kept_after_iteration(R, false)>();
      __syncthreads();
      stage = nstage;
    }
    for (; jt < n_kt; ++jt) {
      const int nstage = stage == NS - 1 ? 0 : stage + 1;
      const bool issued = jt + R.issue_ahead < n_kt;
      if (issued) issue_tile(jt + R.issue_ahead);
      const uint32_t rm = rm_lane + stage * kStageBytes, tr = tr_lane + stage * kStageBytes;
      if constexpr (PARTS == 2) {
        if (2 * jt + part < n_act) step(IC<1>{}, bounded_c, tr, 0, BK * jt + 32 * part, rm_lane + nstage * kStageBytes, 0);
      } else if constexpr (kBlocksPerTile == 2) {
        if (2 * jt < n_act) step(IC<1>{}, bounded_c, tr, 0, BK * jt, rm, 1);
        if (2 * jt + 1 < n_act) step(IC<1>{}, bounded_c, tr, 1, BK * jt + 32, rm_lane + nstage * kStageBytes, 0);
      } else {
        if (jt < n_act) step(IC<1>{}, bounded_c, tr, 0, BK * jt, rm_lane + nstage * kStageBytes, 0);
      }
      if (issued) wait_vmcnt<ring::loads_kept_after_iteration(R, true)>(); else wait_vmcnt<ring::loads_kept_after_iteration(R, false)>();
      __syncthreads();
      stage = nstage;
    }
  };
  if (bounded) run(IC<1>{}); else run(IC<0>{});

  if constexpr (PARTS == 2) {
    // The ring is idle (every wave has passed the last iteration's barrier): part 1 leaves its state there, 16 (8) bytes
    // per lane and access, one slot per wave, and part 0 takes it over.
    constexpr int kSlot = MB * 4096;
    static_assert(2 * kSlot + 2 * 512 <= R.merge_stages * kStageBytes, "two slots in the ring");
    char* const slots = lds + R.merge_stage_first * kStageBytes;
    char* const slot = slots + row_wave * kSlot + lane * 16;
    float2* const stat = reinterpret_cast<float2*>(slots + 2 * kSlot + row_wave * 512) + lane;
    if (part == 1) {
#pragma unroll
      for (int mb = 0; mb < MB; ++mb)
#pragma unroll
        for (int c = 0; c < 4; ++c)
          *reinterpret_cast<f32x4*>(slot + (4 * mb + c) * 1024) = f32x4{oacc[mb][0][4 * c], oacc[mb][0][4 * c + 1], oacc[mb][0][4 * c + 2], oacc[mb][0][4 * c + 3]};
      *stat = make_float2(m_ref[0], l_run[0][0] + l_run[0][1]);
    }
    __syncthreads();
    if (part == 1) return;
    const float2 ml = *stat;
    const float m = fmaxf(m_ref[0], ml.x);
    // both references are 0 on the bounded path; a part without a visible key of the row has (-inf, 0): weight 0
    const float w0 = bounded ? 1.f : fast_exp2(m_ref[0] - m), w1 = bounded ? 1.f : fast_exp2(ml.x - m);
    m_ref[0] = m;
    l_run[0][0] = w0 * (l_run[0][0] + l_run[0][1]) + w1 * ml.y;
    l_run[0][1] = 0.f;
#pragma unroll
    for (int mb = 0; mb < MB; ++mb)
#pragma unroll
      for (int c = 0; c < 4; ++c) {
        const f32x4 t = *reinterpret_cast<const f32x4*>(slot + (4 * mb + c) * 1024);
#pragma unroll
        for (int i = 0; i < 4; ++i) oacc[mb][0][4 * c + i] = w0 * oacc[mb][0][4 * c + i] + w1 * t[i];
      }
  }

  // ---- epilogue: normalise, gate, store y (bf16) and lse (fp32, natural log)
#pragma unroll
  for (int nb = 0; nb < NQB; ++nb) {
    const int row = qw0 + 32 * nb + ln;
    const bool live = row < p.Sq;
    const float l = half_sum(l_run[nb][0] + l_run[nb][1]);
    if (SPLIT && all_kt > a.fwd_chunk) {
      if (live) {
        const int64_t at = (((int64_t)b * p.H + h) * a.fwd_splits + share) * p.Sq + row;
#pragma unroll
        for (int mb = 0; mb < MB; ++mb)
#pragma unroll
          for (int q = 0; q < 4; ++q)
            *reinterpret_cast<float4*>(a.fwd_part + at * D + 32 * mb + 8 * q + 4 * hh) =
                make_float4(oacc[mb][nb][4 * q], oacc[mb][nb][4 * q + 1], oacc[mb][nb][4 * q + 2], oacc[mb][nb][4 * q + 3]);
        if (hh == 0) *reinterpret_cast<float2*>(a.fwd_stat + at * 2) = make_float2(m_ref[nb], l);
      }
      continue;
    }
    float f = fast_rcp(l);
    if (p.gate.ptr) {
      const int rc = live ? row : p.Sq - 1;
      const float z = bf16_to_f32(reinterpret_cast<const uint16_t*>(p.gate.ptr)[(int64_t)b * p.gate.stride_b + (int64_t)rc * p.gate.stride_s + (int64_t)h * p.gate.stride_h]);
      f *= p.gate_scale / (1.0f + __expf(-z));
    }
    if (live && hh == 0) p.lse[((int64_t)b * p.H + h) * p.Sq + row] = (m_ref[nb] + __log2f(l)) * kLn2;
    uint16_t* op = live ? row_ptr_mut<uint16_t>(p.o, b, h, row) : nullptr;
#pragma unroll
    for (int mb = 0; mb < MB; ++mb) {
      float val[16];
#pragma unroll
      for (int r = 0; r < 16; ++r) val[r] = oacc[mb][nb][r] * f;
      store_ct_block(op, mb, hh, live, val);
    }
  }
}

// Adds up the shares of the query tiles that were split: D/4 lanes across a row, G groups of them across the shares.
// Few rows want the shares side by side (4608 rows, 16 shares: 8.9 us with G = 1, 6.4 with a wave per row), many rows are
// better off with more rows per wave (73728 rows, 2 shares: 5.2 and 11.4 us).  Fixed order: deterministic.
// Bound by its chain of loads: a lane's first kMergeEarly shares and the gate are one round trip to memory, where statistics, then
// values, then the gate were three (18 / 6 heads, 256 queries, 8192 keys, the whole call: 30.3 -> 29.9 us).
constexpr int kMergeThreads = 256, kMergeFewRows = 8192, kMergeEarly = 4;
template <int D, int G>
__global__ __launch_bounds__(kMergeThreads) void fwd_merge_kernel(KArgs a) {
  const segpt_attn_params& p = a.p;
  using F = FwdShape<D, D != 64>;
  constexpr int LPR = D / 4, RPW = 64 / (LPR * G), kRows = kMergeThreads / 64 * RPW;
  const int lane = threadIdx.x & 63, part = lane % LPR, gi = lane / (LPR * RPW);
  const int i = blockIdx.x * kRows + (threadIdx.x >> 6) * RPW + lane / LPR % RPW;
  const int h = blockIdx.y, b = blockIdx.z;
  if (i >= p.Sq) return;
  int kend = p.Sk;
  if (p.causal) kend = min(p.Sk, i / F::kBQ * F::kBQ + F::kBQ + p.q_start);
  const int n_kt = (kend + F::kBK - 1) / F::kBK, n = (n_kt + a.fwd_chunk - 1) / a.fwd_chunk;
  if (n <= 1) return;  // written by its only share
  const int64_t at = ((int64_t)b * p.H + h) * a.fwd_splits * p.Sq + i;
  const float2* stat = reinterpret_cast<const float2*>(a.fwd_stat) + at;
  const float* o = a.fwd_part + at * D + 4 * part;
  uint16_t gate = 0;
  if (p.gate.ptr)
    gate = reinterpret_cast<const uint16_t*>(p.gate.ptr)[(int64_t)b * p.gate.stride_b + (int64_t)i * p.gate.stride_s + (int64_t)h * p.gate.stride_h];
  auto stat_of = [&](int s) { return stat[(int64_t)s * p.Sq]; };
  auto row_of = [&](int s) { return *reinterpret_cast<const float4*>(o + (int64_t)s * p.Sq * D); };
  // the first shares are requested together, statistics and values
  float2 ml[kMergeEarly];
  float4 t[kMergeEarly];
#pragma unroll
  for (int u = 0; u < kMergeEarly; ++u) {
    const int s = min(gi + G * u, n - 1);  // past the end: the last share once more, unused
    ml[u] = stat_of(s);
    t[u] = row_of(s);
  }
  float m = ml[0].x;
#pragma unroll
  for (int u = 1; u < kMergeEarly; ++u) m = fmaxf(m, ml[u].x);
  for (int s = gi + G * kMergeEarly; s < n; s += G) m = fmaxf(m, stat_of(s).x);
#pragma unroll
  for (int x = LPR * RPW; x < 64; x <<= 1) m = fmaxf(m, __shfl_xor(m, x, 64));
  float l = 0.f, y[4] = {0.f, 0.f, 0.f, 0.f};
  auto add_share = [&](float2 x, float4 v) {
    const float w = fast_exp2(x.x - m);  // a share without a visible key has (-inf, 0): weight 0
    l += w * x.y;
    y[0] += w * v.x; y[1] += w * v.y; y[2] += w * v.z; y[3] += w * v.w;
  };
#pragma unroll
  for (int u = 0; u < kMergeEarly; ++u)
    if (gi + G * u < n) add_share(ml[u], t[u]);
#pragma unroll 4
  for (int s = gi + G * kMergeEarly; s < n; s += G) add_share(stat_of(s), row_of(s));
#pragma unroll
  for (int x = LPR * RPW; x < 64; x <<= 1) {
    l += __shfl_xor(l, x, 64);
#pragma unroll
    for (int e = 0; e < 4; ++e) y[e] += __shfl_xor(y[e], x, 64);
  }
  float f = 1.0f / l;
  if (p.gate.ptr) f *= p.gate_scale / (1.0f + __expf(-bf16_to_f32(gate)));
  if (gi == 0) {
    if (part == 0) p.lse[((int64_t)b * p.H + h) * p.Sq + i] = (m + __log2f(l)) * kLn2;
    const u32x2 w = {pack_bf16x2(y[0] * f, y[1] * f), pack_bf16x2(y[2] * f, y[3] * f)};
    *reinterpret_cast<u32x2*>(row_ptr_mut<uint16_t>(p.o, b, h, i) + 4 * part) = w;
  }
}

template <int D, bool WIDE, int PARTS = 1>
int launch_fwd_t(const KArgs& a, hipStream_t st) {
  const segpt_attn_params& p = a.p;
  constexpr int BQ = FwdShape<D, WIDE, PARTS>::kBQ;
  const dim3 grid((unsigned)wg_grid((p.Sq + BQ - 1) / BQ, p.B, p.Hkv, p.H / p.Hkv, wg_pinned_pairs(p.B, p.Hkv, false)));
  if (p.rope_cos) hipLaunchKernelGGL((fwd_bf16_kernel<D, WIDE, true, false, PARTS>), grid, dim3(kThreadsM), 0, st, a);
  else hipLaunchKernelGGL((fwd_bf16_kernel<D, WIDE, false, false, PARTS>), grid, dim3(kThreadsM), 0, st, a);
  return (int)hipGetLastError();
}

template <int D>
int launch_fwd_split(const KArgs& a, hipStream_t st) {
  constexpr bool WIDE = D != 64;
  using F = FwdShape<D, WIDE>;
  const segpt_attn_params& p = a.p;
  const int n_qt = (p.Sq + F::kBQ - 1) / F::kBQ;
  const dim3 grid((unsigned)wg_grid(n_qt, p.B, p.Hkv, p.H / p.Hkv, wg_pinned_pairs(p.B, p.Hkv, false)), (unsigned)a.fwd_splits);
  if (p.rope_cos) hipLaunchKernelGGL((fwd_bf16_kernel<D, WIDE, true, true, 1>), grid, dim3(kThreadsM), 0, st, a);
  else hipLaunchKernelGGL((fwd_bf16_kernel<D, WIDE, false, true, 1>), grid, dim3(kThreadsM), 0, st, a);
  const int rc = (int)hipGetLastError();
  if (rc) return rc;
  const bool few = (int64_t)p.B * p.H * p.Sq <= kMergeFewRows;
  constexpr int LPR = D / 4, G = 64 / LPR;
  const int rows = few ? kMergeThreads / 64 : kMergeThreads / LPR;
  const dim3 mgrid((unsigned)((p.Sq + rows - 1) / rows), (unsigned)p.H, (unsigned)p.B);
  if (few) hipLaunchKernelGGL((fwd_merge_kernel<D, G>), mgrid, dim3(kMergeThreads), 0, st, a);
  else hipLaunchKernelGGL((fwd_merge_kernel<D, 1>), mgrid, dim3(kMergeThreads), 0, st, a);
  return (int)hipGetLastError();
}

// Number of key tiles of all query tiles of one head, and of its longest one
template <typename F>
void count_tiles(const segpt_attn_params& p, int64_t* total, int* most) {
  const int n_qt = (p.Sq + F::kBQ - 1) / F::kBQ;
  *total = 0; *most = 0;
  for (int t = 0; t < n_qt; ++t) {
    int64_t kend = p.Sk;
    if (p.causal && (int64_t)(t + 1) * F::kBQ + p.q_start < kend) kend = (int64_t)(t + 1) * F::kBQ + p.q_start;
    const int n = (int)((kend + F::kBK - 1) / F::kBK);
    *total += n;
    *most = n > *most ? n : *most;
  }
}

// Splits the keys of a query tile over several workgroups where the query tiles alone leave CUs idle.  A CU computes
// one key tile (128 rows x 64 keys at head_dim 64, 128 x 32 at 128: 2.1 MFLOP) per 0.59 us whether one workgroup
// is resident or two, and everything here counts in that unit.  Cost of a launch: its longest workgroup, or where there
// are more of them than CUs the average load plus a fifth of the longest; storing a partial result adds kStore, the
// second kernel kMerge and its reading time (94 measured launches: 9 % mean deviation).  A call is split when the model says
// 10 % faster: chunks of a long prompt (18 / 6 heads, 256 queries against 8192 keys: 7 shares, 124 -> 33 us; 1024 queries:
// 120 -> 62), small batches of few queries (10 x 8 heads, 45 queries, 5783 keys: 99 -> 48).
template <typename S, typename N>  // S: shape of a split launch, N: of an unsplit one; n_unit: what a tile of N costs
size_t split_plan(const segpt_attn_params& p, double n_unit, int* splits, int* chunk) {
  constexpr double kCUs = 256, kStore = S::kStoreUnits, kMerge = 7.3, kReadPerUnit = 4.4e6;
  const int64_t heads = (int64_t)p.B * p.H;
  const int n_whole = (p.Sq + N::kBQ - 1) / N::kBQ, n_qt = (p.Sq + S::kBQ - 1) / S::kBQ;
  *splits = 1; *chunk = 0;
  if (heads * n_whole >= 2 * kCUs) return 0;
  auto launch = [&](double items, double total, double longest) {
    return items <= kCUs ? longest : std::max(longest, total / kCUs + 0.2 * longest);
  };
  int64_t total;
  int most;
  count_tiles<N>(p, &total, &most);
  const double whole = n_unit * launch((double)(heads * n_whole), (double)(heads * total), most);
  count_tiles<S>(p, &total, &most);
  double best = 0.9 * whole;
  for (int s = 2; s <= 64; ++s) {
    const int c = (most + s - 1) / s;
    if (c < 4) break;
    if ((most + c - 1) / c != s) continue;
    const double items = (double)heads * std::min((double)n_qt * s, (double)total / c + 0.5 * n_qt);  // shorter tiles: fewer shares
    const double read = (double)heads * s * p.Sq * p.D * sizeof(float) / kReadPerUnit;
    const double cost = launch(items, (double)(heads * total) + 2 * kStore * items, c + kStore) + kMerge + read;
    if (cost < best) { best = cost; *splits = s; *chunk = c; }
  }
  return *splits > 1 ? (size_t)heads * *splits * p.Sq * (p.D + 2) * sizeof(float) : 0;
}

bool wide_fwd(const segpt_attn_params& p) { return p.D != 64 || p.Sk > 2048; }

// Waves of a workgroup that share its query rows (launches whose keys are not split over workgroups).  1: four or eight
// 32-row blocks per workgroup, every wave computes all blocks of a key tile.  2: 64 rows, the two 32-key blocks of a tile go
// to two waves: twice as many workgroups, each half as long, for twice the tile loads and barriers per matrix
// instruction.  2 wins while the launch is as long as its longest workgroup, i.e. while the 128-row workgroups leave resident slots
// empty; the more key tiles a row has, the later that ends.  Measured, 1 against 2, us: head_dim 64, 18 / 6 heads, 1 x
// 512 (72 workgroups) 9.8 / 8.2, 4 x 512 (288) 10.7 / 9.3, 6 x 512 (432) 11.7 / 12.9, 2 x 2048 (576) 34.7 / 28.2, 3 x 2048 (864) 39.8 /
// 40.9, 1 x 4096 (576) 66.7 / 50.6; 8 / 8 heads, 1 x 4096 (256) 61.2 / 34.1; head_dim 128 (one workgroup per CU with 64-key
// tiles), 16 / 4 heads, 2 x 512 (128) 13.9 / 10.9, 4 x 512 (256) 14.9 / 16.1, 1 x 2048 (256) 36.7 / 31.2, 2 x 2048 (512) 47 / 60.
// Calls whose softmax keeps a running reference by their flags stay with 1: with 2 each half rounds its probabilities against a
// reference of its own, which moves every output within bf16 rounding, and their results are kept as they are.  It is not a
// matter of accuracy (2.4e-3 to 2.7e-3 from float64 either way) and costs time without QK-norm, 1 against 2: 1 x 512 13.0 / 10.7, 4
// x 512 14.3 / 12.2, 2 x 2048 41 / 35, 8 / 8 heads, 1 x 4096 87 / 39; head_dim 128, 2 x 512 17.8 / 13.4, 1 x 2048 48 / 36.5.
int fwd_parts(const segpt_attn_params& p) {
  if (p.flags & (SEGPT_FLAG_RUNNING_MAX | SEGPT_FLAG_NO_NORM)) return 1;
  const int64_t wgs = (int64_t)p.B * p.H * ((p.Sq + 127) / 128), tiles = (p.Sk + kBK - 1) / kBK;
  if (p.D == 64) return wgs <= (tiles >= 32 ? 640 : 384) ? 2 : 1;
  return wgs <= (tiles >= 16 ? 256 : 128) ? 2 : 1;
}

}  // namespace

// Forward-only calls: bytes of the partials when the keys are to be split, 0 when not.
size_t fwd_split_plan(const segpt_attn_params& p, int* splits, int* chunk) {
  if (p.D == 128) return split_plan<FwdShape<128, true>, FwdShape<128, true>>(p, 1.0, splits, chunk);
  if (wide_fwd(p)) return split_plan<FwdShape<64, false>, FwdShape<64, true>>(p, 1.5, splits, chunk);
  return split_plan<FwdShape<64, false>, FwdShape<64, false>>(p, 1.0, splits, chunk);
}

int launch_fwd_bf16(const KArgs& a, hipStream_t st) {
  if (a.p.D == 64) {
    if (a.fwd_splits > 1) return launch_fwd_split<64>(a, st);
    if (fwd_parts(a.p) == 2) return launch_fwd_t<64, false, 2>(a, st);
    return wide_fwd(a.p) ? launch_fwd_t<64, true>(a, st) : launch_fwd_t<64, false>(a, st);
  }
  if (a.p.D == 128) {
    if (a.fwd_splits > 1) return launch_fwd_split<128>(a, st);
    return fwd_parts(a.p) == 2 ? launch_fwd_t<128, true, 2>(a, st) : launch_fwd_t<128, true>(a, st);
  }
  return (int)hipErrorInvalidValue;
}

}  // namespace segpt
