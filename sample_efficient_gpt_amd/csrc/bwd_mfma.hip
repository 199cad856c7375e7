// bf16 backward: two deterministic MFMA kernels (no floating-point atomics).
//
// Operands are normalised tensors held in the workspace (bf16):
//   Khat = b_j k_j and V' = c1 v + c2 v_first, written by the key/value pre-pass (pre_post.hip);
//   Qhat = sm_scale*log2e * a_i q_i * g_q*g_k and the two row statistics -lse2, -delta (which also carry a positive
//   gate factor), written by the dQ kernel for the dK/dV kernel that runs after it.
//
//  bwd_dq    query-stationary, same orientation as the forward (a lane owns one query column):
//              S^T  = Khat . Qhat^T - lse2        dP^T = V' . dO^T - delta     (A from LDS row-major,
//              dS^T = exp2(S^T) * dP^T            T^T += Khat^T . dS^T          B = registers; the row
//            statistics enter as the MFMA's C operand, so no subtraction is spent on them)
//            epilogue: through the q normaliser, dq (bf16), and this workgroup's partial of the
//            combined scale gradient dg[d] = sum_i sm_scale * (a_i q_id) * T_id.
//  bwd_dkdv  key-stationary (a lane owns one key column); a wave owns 32 keys of one kv head and walks
//            the query tiles of every query head of the group (dK/dV of a GQA group are summed in
//            registers):
//              S  = Qhat . Khat^T - lse2          dP = dO . V'^T - delta
//              dV'^T += dO^T . P                  dKhat^T += Qhat^T . dS        (A = transposing LDS read)
//            epilogue: through the k normaliser, dk, dv (= c1 dV'), dv_first (= c2 dV'), (dc1, dc2) partials.
//
// One workgroup = 4 waves (one per SIMD); at head_dim 64 two workgroups share a CU so that the softmax-like VALU
// phase of one overlaps the MFMA phase of another.  Streamed tiles (64 rows) travel through a ring in LDS.  Both kernels
// have a second form of their loop (PIPE) in which a wave overlaps the two phases by itself: dkdv_pipelined(), dq_pipelined().
#include "mfma_common.hpp"
#include "ring_protocol.hpp"

namespace segpt {

int bf16_dq_grid(const segpt_attn_params& p);
int bf16_dkdv_grid(const segpt_attn_params& p);

namespace {

constexpr int kBwdRows = 4 * 32;  // rows (queries for dQ, keys for dK/dV) owned by a workgroup

// The dK/dV launch pins (batch, kv head) pairs to XCDs only when ALL of them can be pinned: with a spread remainder it
// was measured 13 % slower at B*Hkv = 12, S = 8192 (where forward and dQ gain 2-4 % from pinning 8 of the 12).
__host__ __device__ inline int dkdv_pinned(const segpt_attn_params& p) { return wg_pinned_pairs(p.B, p.Hkv, true); }

// How the four waves of a dK/dV workgroup share a launch's work.  1: four key blocks (128 keys), every wave computes both
// 32-query blocks of a streamed tile.  2: two key blocks (64 keys) times the two query blocks of the tile: twice as many
// workgroups, each half as long, for twice the tile loads and barriers per matrix instruction.  What decides is whether
// the launch is as long as its longest workgroup (the early key tiles stream every query of every head of the group) or
// as its total work, i.e. how many 128-key workgroups there are for the 512 (head_dim 64, two per CU) or 256 (head_dim
// 128) resident ones.  Measured, 1 against 2, us: head_dim 64, 18 / 6 heads, 1 x 2048 (96 workgroups) 100 / 63, 8 x 999 (384)
// 71 / 57, 1 x 8192 (384) 430 / 318, 6 x 2048 (576) 132 / 126, 8 x 2048 (768) 156 / 160; head_dim 128, 16 / 4 heads,
// 4 x 2048 (256) 226 / 151, 6 x 2048 (384) 235 / 237, 8 x 2048 (512) 272 / 302.  Between half full and full, short
// workgroups (8 / 8 heads, 12 x 512, 8 tiles each: 17.1 / 17.6) have too little to halve: kLongTiles and more do (16 x 512,
// 18 / 6 heads, 24 tiles: 34.8 / 32.2).
inline int dkdv_parts(const segpt_attn_params& p) {
  constexpr int kLongTiles = 24;
  const int64_t wgs = (int64_t)p.B * p.Hkv * ((p.Sk + kBwdRows - 1) / kBwdRows);
  const int64_t tiles = (int64_t)(p.H / p.Hkv) * ((p.Sq + kBK - 1) / kBK);
  return wgs <= 256 || (p.D == 64 && wgs <= 512 && tiles >= kLongTiles) ? 2 : 1;
}

// The same for the query rows of a dQ workgroup: 1: 128 rows, 2: 64 rows times the two 32-key blocks of a tile.  Both waves of
// a pair compute the row prologue (normaliser, Qhat, delta), so 2 costs more here and ends earlier.  Measured, 1 against 2,
// us: head_dim 64, 18 / 6 heads, 2 x 512 (144 workgroups) 12.1 / 10.3, 4 x 512 (288) 13.9 / 16.2, 1 x 2048 (288) 32.3 / 25.1;
// 16 / 4 heads, 4 x 512 (256) 13.2 / 11.5, 3 x 1024 (384) 21.9 / 21.9, 1 x 4096 (512) 67 / 66; head_dim 128, 2 x 512 (128) 19.6 /
// 16.4, 3 x 512 (192) 21.0 / 23.1, 2 x 1024 (256) 31.4 / 32.3.
inline int dq_parts(const segpt_attn_params& p) {
  constexpr int kLongTiles = 16;
  const int64_t wgs = (int64_t)p.B * p.H * ((p.Sq + kBwdRows - 1) / kBwdRows), tiles = (p.Sk + kBK - 1) / kBK;
  return wgs <= (p.D == 128 ? 128 : tiles >= kLongTiles ? 384 : 256) ? 2 : 1;
}

// Whether a launch of 128-row workgroups takes the kernel whose loop is laid out instruction by instruction (PIPE).  Its start and end
// cost a workgroup a few hundred cycles more (a block's scores that nothing overlaps, a tile that is requested once too often).
// head_dim 64, us, compiler's loop / PIPE, causal plain calls.  dK/dV, 18 / 6 heads, 16384 tokens in all: at 256 / 512 / 768 / 999 / 1536 / 3072 tokens
// (12 / 24 / 36 / 48 / 72 / 144 streamed tiles) 42.1 / 42.1, 61.0 / 56.4, 75.3 / 75.7, 96.2 / 93.2, 121.8 / 115.2, 239.2 / 207.8; other heads at 48 tiles:
// 8 / 8, 5 x 3072 110.7 / 103.1, 16 / 4, 32 x 768 95.1 / 94.4 (not causal 164.4 / 148.3), 16 / 2, 96 x 384 83.7 / 79.6.  dQ, 18 / 6 heads: at 256 / 768 / 1152 /
// 2048 / 3072 (4 / 12 / 18 / 32 / 48 tiles) 55.0 / 55.6, 73.0 / 70.4, 89.6 / 87.6, 138.6 / 128.8, 180.6 / 167.6, with a rotary embedding 59.9 / 61.2,
// 81.4 / 79.2, 97.7 / 94.2, 143.9 / 135.2, 184.4 / 173.8; 8 / 8, 8 x 2048 65.6 / 62.7 (not causal 109.6 / 103.8).  The lines were drawn when dK/dV still
// computed masked blocks; below them PIPE now wins at some shapes (dK/dV 16 / 4, 64 x 384 65.6 / 61.1, 8 / 8, 16 x 1024 50.1 / 47.3) and loses or
// is even at others (above; dQ 16 / 2, 192 x 192 117.9 / 122.9).
// head_dim 128 has one wave per SIMD and nothing else to fill the matrix pipe with: always.  dQ and dK/dV, 16 / 4 heads: 96 x 256 201.6 / 199.1 and 117.6 /
// 112.1 (not causal 216.4 / 220.3 and 162.9 / 142.9), 24 x 1024 298.9 / 282.1 and 258.8 / 204.9, 12 x 2048 430.1 / 402.9 and 477.2 / 372.7; 8 / 8, 48 x 256
// 57.1 / 54.3 and 52.2 / 52.0, 6 x 2048 113.2 / 101.7 and 139.0 / 113.5.
inline bool dkdv_pipelined(const segpt_attn_params& p) {
  constexpr int kTiles = 48;
  return dkdv_parts(p) == 1 && (p.D == 128 || (int64_t)(p.H / p.Hkv) * ((p.Sq + kBK - 1) / kBK) >= kTiles);
}
inline bool dq_pipelined(const segpt_attn_params& p) {
  constexpr int kTiles = 32;
  return dq_parts(p) == 1 && (p.D == 128 || (p.Sk + kBK - 1) / kBK >= kTiles);
}

constexpr float kGateFactorFloor = 1e-30f;  // a smaller gate factor switches its row off in the dK/dV kernel

constexpr int kStages = 4;  // LDS ring of streamed stages (two tiles each): tile t lives in stage t % 4

// ============================================================================================ dQ
// Also the producer of the per-query-row quantities the dK/dV kernel streams afterwards: Qhat, -delta,
// -lse*log2e and (with a gate) dgate; the gate-scaled copy of dO only when the gate scale is not positive.
//
// Software pipeline over 32-key blocks n (two per staged tile), one barrier per tile:
//   B(n)  S^T, dP^T MFMAs from the row-major fragments requested one block earlier
//   C(n)  request the transposed Khat fragments of block n
//   D(n)  dS^T = exp2(S^T) * dP^T, pack to bf16
//   A(n+1) request the row-major fragments of block n+1 (possibly the next tile, already in LDS)
//   E(n)  T^T += Khat^T dS^T MFMAs
// Tiles travel global->LDS directly (no registers), three tiles ahead of their use.
// ROPE (rope tables given) is a compile-time switch so that the table rows are ordinary, unconditional loads which
// travel with the start-up tiles (prologue) and with the first stores (epilogue) instead of costing a memory round
// trip of their own behind a branch.
//
// PARTS: see dq_parts(); with 2 the workgroup owns 64 query rows, two waves each take one of the two 32-key blocks of
// every tile for the same rows, and the pair adds up T^T through LDS behind the loop.
// PIPE (PARTS == 1): see dq_pipelined().
template <int D, bool ROPE, int PARTS, bool PIPE>
__global__ __launch_bounds__(kThreadsM, D == 64 ? 2 : 1) void bwd_dq_bf16_kernel(KArgs a) {
  using Z = Swz<D>;
  static_assert(PARTS == 1 || (PARTS == 2 && !PIPE), "a tile has two 32-key blocks");
  constexpr int BQ = kBwdRows / PARTS;
  constexpr int kRowWaves = 4 / PARTS;  // waves side by side along the query rows
  constexpr int KS = D / 16;
  constexpr int MB = D / 32;
  constexpr int kStageBytes = 2 * Z::kTileBytes;
  // the pipeline's numbers: ring_protocol.hpp
  constexpr bool AGPR = D == 128;
  constexpr ring::Protocol R = PARTS == 1 ? (ROPE ? ring::dq_rope(Z::kPasses, PIPE) : ring::dq(Z::kPasses, PIPE))
                                          : (ROPE ? ring::dq_rope_parts(Z::kPasses) : ring::dq_parts(Z::kPasses));
  static_assert(ring::well_formed(R) && R.stages == kStages && !R.issue_at_top, "tile pipeline");
  static_assert(ROPE ? (R.pre_row_stages == 4 && R.row_stages == 1 && R.early_tiles == R.startup_tiles && !R.wait_before_loop && R.epilogue_row_stages == (PARTS == 1 ? 2 : 1))
                     : (R.pre_row_stages == 0 && R.row_stages == 3 && R.wait_before_loop && R.epilogue_row_stages == 0), "tile pipeline");
  const segpt_attn_params& p = a.p;
  __shared__ __attribute__((aligned(1024))) char lds[kStages * kStageBytes];
  __shared__ __attribute__((aligned(16))) float gsm[D];       // g_q * g_k, read as float4 slices
  constexpr int kRedStride = D + 4;                 // floats per row of the dg staging area (16-byte aligned rows)
  constexpr int kColGroups = D / 4;                 // a thread sums 4 adjacent columns ...
  constexpr int kRowGroups = kThreadsM / kColGroups;  // ... over one of these groups of rows
  constexpr int kRowsPerGroup = BQ / kRowGroups;
  __shared__ __attribute__((aligned(16))) float red4[kRowGroups * D];  // per-row-group column sums of the dg partial
  static_assert(kStages * kStageBytes >= BQ * kRedStride * 4, "LDS reuse for the dg partial");

  const int tid = threadIdx.x, lane = tid & 63;
  const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);  // wave-uniform: everything derived from it stays scalar
  const int ln = lane & 31, hh = lane >> 5;
  const int rep = p.H / p.Hkv;
  const int n_qt = (p.Sq + BQ - 1) / BQ;
  const WgCoord wg = decode_wg(D == 64 ? balanced_id(blockIdx.x, gridDim.x) : (int)blockIdx.x, n_qt, p.B, p.Hkv, rep, wg_pinned_pairs(p.B, p.Hkv, false));
  if (!wg.valid) {  // idle padding workgroup: its row of the scale-gradient partials must still read as zero
    if (tid < D) a.dg_part[(int64_t)blockIdx.x * D + tid] = 0.f;
    return;
  }
  const int b = __builtin_amdgcn_readfirstlane(wg.b), g = __builtin_amdgcn_readfirstlane(wg.g);  // divided in vector registers
  const int h = __builtin_amdgcn_readfirstlane(wg.g * rep + wg.hh);
  const int q0 = __builtin_amdgcn_readfirstlane(wg.tile) * BQ;
  const int row_wave = PARTS == 1 ? wave : wave % kRowWaves, part = PARTS == 1 ? 0 : wave / kRowWaves;
  const int qw0 = q0 + row_wave * 32;
  const int row = qw0 + ln;
  const bool live = row < p.Sq;
  const int row_c = live ? row : p.Sq - 1;  // padding lanes recompute the last row and store nothing
  const int64_t head_row = ((int64_t)b * p.H + h) * p.Sq;  // scalar: what the epilogue needs of it costs no vector registers over the loop

  int kend = p.Sk;
  if (p.causal) kend = min(p.Sk, q0 + BQ + p.q_start);
  const int n_kt = (kend + kBK - 1) / kBK;
  const char* kbase = reinterpret_cast<const char*>(a.khat + ((int64_t)b * p.Hkv + g) * p.Sk * D);
  const char* vbase = a.vmix ? reinterpret_cast<const char*>(a.vmix + ((int64_t)b * p.Hkv + g) * p.Sk * D)
                             : reinterpret_cast<const char*>(row_ptr<uint16_t>(p.v, b, g, 0));
  const uint32_t kstep = D * 2, vstep = a.vmix ? (uint32_t)D * 2 : (uint32_t)p.v.stride_s * 2;

  const uint32_t lds0 = lds_addr_of(lds);
  const int2 src = swz_src<D>(lane, wave);
  const uint32_t wave_dst = lds0 + wave * 1024;
  const TileLaneOff<D> full_tile = tile_lane_offsets<D>(kstep, vstep, kBK, src.x, src.y);
  auto issue_tile = [&](int jt) {  // tile jt -> stage jt % kStages
    const char* ksrc = kbase + (int64_t)jt * kBK * kstep;
    const char* vsrc = vbase + (int64_t)jt * kBK * vstep;
    const uint32_t dst = wave_dst + (jt % kStages) * kStageBytes;
    const int left = p.Sk - jt * kBK;
    if (left >= kBK) issue_tile_pair<D>(ksrc, vsrc, full_tile, dst);
    else issue_tile_pair<D>(ksrc, vsrc, tile_lane_offsets<D>(kstep, vstep, left, src.x, src.y), dst);
  };

  // ---- The workgroup's 128 query / dO / output rows come in as tiles too: read row-per-lane from global memory
  // every wave-wide load would touch 32 cache lines for 32 bytes each and the prologue would spend its time in
  // the address path of the vector memory unit; staged through LDS by direct loads they are whole lines, and the
  // row-major fragment read of a tile is exactly the B-operand layout (lane = row, 8 entries of k-step ks).
  // Without a rotary embedding: stage 0 takes key tile 0; stages 1..3 hold the q, dO and o blocks until the rows sit
  // in registers, then key tiles 1 and 2 are requested into stages 1 and 2 and the ring turns as usual.  All of it
  // is in flight at once, with the row's lse, the gate logit and the scale vector behind it: one memory round trip
  // (vector-memory waits are in order, and the compiler's own count does not see the direct loads, so its first
  // wait covers them).
  // With a rotary embedding the table rows of the 128 positions (D/2 floats: as long as a tensor row) are two more
  // blocks, for the same reason, and the start-up has two phases: q, cos, sin, dO in stages 0..3; once they are in
  // registers, the o block in stage 3 and key tiles 0..2 in stages 0..2, which arrive while Qhat is computed.
  // The prologue's results (Qhat, gated dO, -delta, -lse2, dgate) are stored from the epilogue, so no store is in
  // flight while the loop counts its tile loads.
  constexpr int kRowStage = R.row_stage_first;
  constexpr int kQStage = ROPE ? 0 : kRowStage, kCosStage = 1, kSinStage = 2;
  constexpr int kDoStage = ROPE ? 3 : kRowStage + 1, kOStage = ROPE ? kRowStage : kRowStage + 2;
  static_assert(!ROPE || kOStage == 3, "first phase: q, cos, sin, dO; second phase: tiles 0..2, o");
  // where the row blocks lie.  PARTS == 2: blocks of 64 rows, two of them are the two tiles of one stage
  constexpr uint32_t kPair = Z::kTileBytes;
  constexpr uint32_t kQRows = kQStage * kStageBytes, kDoRows = PARTS == 1 ? kDoStage * kStageBytes : kQRows + kPair;
  constexpr uint32_t kCosRows = kCosStage * kStageBytes, kSinRows = PARTS == 1 ? kSinStage * kStageBytes : kCosRows + kPair;
  constexpr uint32_t kORows = kOStage * kStageBytes;
  const int rows_left = min(p.Sq - q0, BQ);
  const char* qb = reinterpret_cast<const char*>(row_ptr<uint16_t>(p.q, b, h, q0));
  const char* db = reinterpret_cast<const char*>(row_ptr<uint16_t>(p.d_o, b, h, q0));
  const char* yb = reinterpret_cast<const char*>(row_ptr<uint16_t>(p.o, b, h, q0));
  const int64_t rope_row0 = ROPE ? (int64_t)(p.rope_q_pos0 + q0) * (D / 2) : 0;  // the tables' row of query q0
  const uint32_t qst = (uint32_t)p.q.stride_s * 2, dst = (uint32_t)p.d_o.stride_s * 2, yst = (uint32_t)p.o.stride_s * 2;
  auto issue_rope_rows = [&](uint32_t cos_at, uint32_t sin_at) {  // BQ table rows each, laid out like tensor rows
    const char* cb = reinterpret_cast<const char*>(p.rope_cos + rope_row0);
    const char* sb = reinterpret_cast<const char*>(p.rope_sin + rope_row0);
    if constexpr (PARTS == 1) {
      const TileLaneOff<D> o = rowblock_lane_offsets<D>(D * 2, 0, rows_left, src.x, src.y);
      issue_tile_pair<D>(cb, cb, o, wave_dst + cos_at);
      issue_tile_pair<D>(sb, sb, o, wave_dst + sin_at);
    } else {
      issue_tile_pair<D>(cb, sb, tile_lane_offsets<D>(D * 2, D * 2, rows_left, src.x, src.y), wave_dst + cos_at);
    }
  };
  auto issue_o_rows = [&]() {
    if constexpr (PARTS == 1) issue_tile_pair<D>(yb, yb, rowblock_lane_offsets<D>(yst, 0, rows_left, src.x, src.y), wave_dst + kORows);
    else issue_tile_pair<D>(yb, yb, tile_lane_offsets<D>(yst, yst, rows_left, src.x, src.y), wave_dst + kORows);
  };
  if constexpr (!ROPE) {
#pragma unroll
    for (int t = 0; t < R.early_tiles; ++t)
      if (t < n_kt) issue_tile(t);
  }
  if constexpr (PARTS == 1) {
    issue_tile_pair<D>(qb, qb, rowblock_lane_offsets<D>(qst, 0, rows_left, src.x, src.y), wave_dst + kQRows);
    if constexpr (ROPE) issue_rope_rows(kCosRows, kSinRows);
    issue_tile_pair<D>(db, db, rowblock_lane_offsets<D>(dst, 0, rows_left, src.x, src.y), wave_dst + kDoRows);
  } else {
    issue_tile_pair<D>(qb, db, tile_lane_offsets<D>(qst, dst, rows_left, src.x, src.y), wave_dst + kQRows);
    if constexpr (ROPE) issue_rope_rows(kCosRows, kSinRows);
  }
  if constexpr (!ROPE) issue_o_rows();
  const float lse_row = (p.lse + head_row)[row_c];
  // the conditional reads last: the compiler waits for every outstanding load where their branches join
  float gate_z = 0.f;
  if (p.gate.ptr)
    gate_z = bf16_to_f32(reinterpret_cast<const uint16_t*>(p.gate.ptr)[(int64_t)b * p.gate.stride_b + (int64_t)row_c * p.gate.stride_s + (int64_t)h * p.gate.stride_h]);
  float gval = 0.f;
  if (tid < D) gval = gprod_at(p, tid);
  if (tid < D) gsm[tid] = gval;
  wait_vmcnt<0>();
  __syncthreads();
  // rows 32*row_wave .. +31 of a block: half (row_wave >> 1) of it, row block (row_wave & 1) of that tile
  u32x4 qraw[KS], dyraw[KS], yraw[KS];
  u32x2 qct[MB][4];  // the query row once more, in the layout of the epilogue's C tiles (packed pairs)
  RopeB<KS> rope_b;
  const uint32_t row_half = (row_wave >> 1) * Z::kTileBytes, row_rb = row_wave & 1;
  const uint32_t row_rm = lds0 + row_half + swz_off_rm<D>(lane);
  const uint32_t row16 = lds0 + row_half + swz_off_row16<D>(lane) + row_rb * 32 * Z::kRB;  // chunk 0 of the lane's row
  {
    const uint32_t ct = lds0 + kQRows + row_half + swz_off_ct<D>(lane) + row_rb * 32 * Z::kRB;
#pragma unroll
    for (int ks = 0; ks < KS; ++ks) {
      qraw[ks] = __builtin_bit_cast(u32x4, swz_frag_rm<D>(row_rm + kQRows, row_rb, ks));
      dyraw[ks] = __builtin_bit_cast(u32x4, swz_frag_rm<D>(row_rm + kDoRows, row_rb, ks));
      if constexpr (!ROPE) yraw[ks] = __builtin_bit_cast(u32x4, swz_frag_rm<D>(row_rm + kORows, row_rb, ks));
    }
#pragma unroll
    for (int mb = 0; mb < MB; ++mb)
#pragma unroll
      for (int c = 0; c < 4; ++c) qct[mb][c] = lds_read8(ct ^ (uint32_t)((4 * mb + c) << 4));
    if constexpr (ROPE) rope_b = rope_b_from_lds<KS>(row16 + kCosRows, row16 + kSinRows, hh);
  }
  __syncthreads();  // the borrowed stages are free again
  if constexpr (ROPE) {
    issue_o_rows();
#pragma unroll
    for (int t = 0; t < R.early_tiles; ++t)
      if (t < n_kt) issue_tile(t);
  } else {
#pragma unroll
    for (int t = R.early_tiles; t < R.startup_tiles; ++t)
      if (t < n_kt) issue_tile(t);
  }

  // ---- query-row prologue: alpha, Qhat, delta, gate; B operands stay in registers
  bf16x8 qreg[KS], doreg[KS];
  float alpha, delta, dgate_row = 0.f, gfac = 1.f, gate_sg = 0.f;
  auto row_dot = [&]() {  // delta = rowsum(dY * Y): the o block is the last thing the second phase waits for
    float dl = 0.f;
#pragma unroll
    for (int ks = 0; ks < KS; ++ks)
#pragma unroll
      for (int i = 0; i < 4; ++i) dl += bf16lo(yraw[ks][i]) * bf16lo(dyraw[ks][i]) + bf16hi(yraw[ks][i]) * bf16hi(dyraw[ks][i]);
    delta = half_sum(dl);
    if (p.gate.ptr) dgate_row = (1.0f - gate_sg) * delta;
  };
  if (p.gate.ptr) {
    gate_sg = 1.0f / (1.0f + __expf(-gate_z));
    gfac = p.gate_scale * gate_sg;
  }
  if constexpr (!ROPE) row_dot();
  {
    float qx[KS][8];
    unpack_b_layout<KS>(qraw, qx);
    if (ROPE) rope_b_apply<KS>(qx, rope_b);
    float ss = 0.f;
#pragma unroll
    for (int ks = 0; ks < KS; ++ks)
#pragma unroll
      for (int t = 0; t < 8; ++t) ss += qx[ks][t] * qx[ks][t];
    ss = half_sum(ss);
    alpha = row_normaliser_fast(p, ss, 1.0f / D);
    const float f = alpha * p.sm_scale * kLog2e;
#pragma unroll
    for (int ks = 0; ks < KS; ++ks) {
      const float4 ga = *reinterpret_cast<const float4*>(gsm + 16 * ks + 8 * hh);
      const float4 gb = *reinterpret_cast<const float4*>(gsm + 16 * ks + 8 * hh + 4);
      u32x4 w;
      w[0] = pack_bf16x2(qx[ks][0] * f * ga.x, qx[ks][1] * f * ga.y);
      w[1] = pack_bf16x2(qx[ks][2] * f * ga.z, qx[ks][3] * f * ga.w);
      w[2] = pack_bf16x2(qx[ks][4] * f * gb.x, qx[ks][5] * f * gb.y);
      w[3] = pack_bf16x2(qx[ks][6] * f * gb.z, qx[ks][7] * f * gb.w);
      qreg[ks] = as_bf16x8(w);
      doreg[ks] = as_bf16x8(p.gate.ptr ? scale8(dyraw[ks], gfac) : dyraw[ks]);
    }
  }
  if constexpr (ROPE) {
    // second phase landed (tile 2 with it: no late tile, no further wait before the loop); the o rows go to registers
    // and one more barrier frees their stage, which iteration 0 refills
    wait_vmcnt<0>();
    __syncthreads();
#pragma unroll
    for (int ks = 0; ks < KS; ++ks) yraw[ks] = __builtin_bit_cast(u32x4, swz_frag_rm<D>(row_rm + kORows, row_rb, ks));
    row_dot();
    __syncthreads();
  }
  // row statistics as MFMA C operands (every register of a lane belongs to the lane's query); the dK/dV
  // kernel reads the same two numbers per row from the workspace
  const float nlse2 = -lse_row * kLog2e;
  const f32x16 c_lse = splat16(nlse2);
  const f32x16 c_del = splat16(-delta);

  f32x16 acc[MB];
#pragma unroll
  for (int mb = 0; mb < MB; ++mb) acc[mb] = splat16(0.f);

  // blocks this wave has to visit (causal: up to the block holding its last query's diagonal)
  int n_act = (kend + 31) / 32;
  if (p.causal) n_act = min(n_act, (qw0 + 31 + p.q_start) / 32 + 1);
  const int qlim = p.causal ? min(row + p.q_start, p.Sk - 1) : p.Sk - 1;  // last visible key of this lane's query

  // PARTS == 2: this wave's block of every tile is number `part` (a multiple of 4 KB further: the XOR terms stay below)
  const uint32_t rm_lane = lds0 + swz_off_rm<D>(lane) + part * 32 * Z::kRB;
  const uint32_t tr_lane = lds0 + swz_off_tr<D>(lane) + part * 32 * Z::kRB;
  bf16x8 kf[KS], vf[KS];
  // ---- pipeline start-up.  Every iteration of the loop starts with its own tile AND the next one landed (the
  // second block of a tile already requests the next tile's fragments) and at most one more in flight, so tile 1,
  // requested after the row blocks had left its stage, must be complete here; the row prologue above ran in
  // between, so this wait is short.  Tile 2 stays in flight.
  if constexpr (R.wait_before_loop) {
    if (n_kt >= R.startup_tiles) wait_vmcnt<ring::loads_kept_before_loop(R, R.startup_tiles)>(); else wait_vmcnt<0>();
    __syncthreads();
  }
  // leading blocks of this wave that need no mask (every key visible to every query of the wave, inside Sk)
  int n_full = p.Sk / 32;
  if (p.causal) n_full = min(n_full, (qw0 + p.q_start + 1) / 32);
  // Loop A: tiles whose two blocks need no mask; loop B: the rest (masking a fully visible block is a no-op).
  // Two loops, so that each body holds one variant of the block and the accumulators never meet at a join.
  const int n_a = PARTS == 1 ? n_full / 2 : (n_full + 1 - part) / 2;  // n_full <= n_act
  if constexpr (PIPE) {
    // The pipeline of the dK/dV kernel below (there: what a slot holds, and why): step n computes S^T and dP^T of block n + 1
    // (kA matrix instructions) while the vector unit turns those of block n into dS^T, then adds block n to T^T (kB);
    // the row-major fragments of block n + 2 come in as those of block n + 1 are used.
    // dQ, us: head_dim 128, 4 x 16 / 4 heads, 4096 tokens 452 -> 406 (942 k -> 770 k cycles, matrix pipe 42 -> 52 % busy; a quarter
    // of the launch is now the workgroups' first and last thousands of cycles, one workgroup a CU); head_dim 64, 2 x 18 / 6
    // heads, 8192 tokens 437 -> 421 (775 k -> 692 k cycles, 57 -> 64 % busy, 1.78 -> 1.65 GHz).  At head_dim 64
    // everything is in ordinary registers (248 of 256, 255 with a rotary embedding): a kernel that uses both files gets half of each, and the ordinary
    // half spills.
    constexpr int kA = 2 * KS, kB = 2 * MB;
    auto order = [](int i) { return (i & 1) * KS + (i >> 1); };  // i-th product: k-step of S^T, or KS + that of dP^T
    f32x16 s0, d0, s1, d1;           // scores and dP of two consecutive blocks
    uint32_t rma[KS], tra[2 * MB];   // addresses: the next tile's row-major fragments, this tile's transposed ones
    auto start = [&](f32x16& s, f32x16& d, int i) {  // the i-th product of a block
      const int o = order(i), ks = o % KS;
      if (o >= KS) ks == 0 ? mfma32_fixed_from<AGPR>(d, vf[ks], doreg[ks], c_del) : mfma32_fixed<AGPR>(d, vf[ks], doreg[ks]);
      else ks == 0 ? mfma32_fixed_from<AGPR>(s, kf[ks], qreg[ks], c_lse) : mfma32_fixed<AGPR>(s, kf[ks], qreg[ks]);
    };
    auto row_frag = [&](uint32_t rm_ks, int kb, int o) { (o < KS ? kf : vf)[o % KS] = as_bf16x8(lds_read16(rm_ks + (o < KS ? 0 : Z::kTileBytes) + kb * 32 * Z::kRB)); };
    // (s, d): block n, whose first key is jb, number kb of its tile; (sn, dn): block n + 1.  mem and alu: what else the slots
    // hold, beside the LDS reads and beside the vector instructions
    // masked_c: 0 no mask, 1 masked, 2 masked and the wave's last block (no products of a next one, whose registers would be
    // given to others while they are still on their way)
    auto step = [&](auto masked_c, f32x16& s, f32x16& d, f32x16& sn, f32x16& dn, int kb, int jb, auto mem, auto alu) {
      constexpr bool MASKED = decltype(masked_c)::value != 0, LAST = decltype(masked_c)::value == 2;
      // register r holds key jb + 4hh + c_r, c_r = 8(r/4) + r%4: masked iff c_r > qlim - jb - 4hh
      const int t = qlim - jb - 4 * hh;
      u32x4 dw[2];  // dS as operand, in halves of 16 keys
      bf16x8 kT[MB][2];
      auto v_exp = [&](int r) {
        if (MASKED && 8 * (r >> 2) + (r & 3) > t) s[r] = -INFINITY;
        s[r] = fast_exp2(s[r]);
      };
      auto v_mul = [&](int r) { s[r] *= d[r]; };
      auto v_ds = [&](int j) { dw[j >> 2][j & 3] = pack_bf16x2(s[2 * j], s[2 * j + 1]); };
      constexpr int kExps = 16 / kA;  // per slot
#pragma unroll
      for (int i = 0; i < kA; ++i) {
        if constexpr (!LAST) start(sn, dn, i);
        // even slots: a transposed fragment of block n; odd ones: a row-major fragment of block n + 2, whose place is free
        if (i & 1) { if constexpr (!LAST) row_frag(rma[order(i >> 1) % KS], kb, order(i >> 1)); }
        else kT[(i >> 1) % MB][(i >> 1) / MB] = frag_tr_at<D>(tra[2 * ((i >> 1) % MB)], tra[2 * ((i >> 1) % MB) + 1], 2 * kb + (i >> 1) / MB, 0);
        mem(i);
        __builtin_amdgcn_sched_barrier(0);
#pragma unroll
        for (int e = 0; e < kExps; ++e) {
          const int r = kExps * i + e;
          v_exp(r);
          if (r >= kExps) v_mul(r - kExps);
          if (r >= kExps + 2 && (r - kExps) % 2 == 0) v_ds((r - kExps) / 2 - 1);
        }
        if (i == kA - 1) {
#pragma unroll
          for (int r = 16 - kExps; r < 16; ++r) v_mul(r);
#pragma unroll
          for (int j = 8 - kExps; j < 8; ++j) v_ds(j);
        }
        alu(i);
        __builtin_amdgcn_sched_barrier(0);
      }
#pragma unroll
      for (int j = 0; j < kB; ++j) {
        mfma32_acc<AGPR>(acc[j % MB], kT[j % MB][j / MB], as_bf16x8(dw[j / MB]));
        if constexpr (!LAST) row_frag(rma[order(kA / 2 + j) % KS], kb, order(kA / 2 + j));
        mem(kA + j);
        __builtin_amdgcn_sched_barrier(0);
        alu(kA + j);
        __builtin_amdgcn_sched_barrier(0);
      }
    };
    static_assert(kB == kA / 2, "one row-major fragment per slot of the second half, the others in the odd ones of the first");
    auto rm_addr = [&](uint32_t rm, int ks) { return rm ^ (uint32_t)(ks << 5); };
    auto tr_addr = [&](uint32_t tr, int x) { return tr ^ (uint32_t)(((x >> 1) << 6) ^ (x & 1 ? Z::kHiXor : 0)); };
#pragma unroll
    for (int ks = 0; ks < KS; ++ks) rma[ks] = rm_addr(rm_lane + kStageBytes, ks);
#pragma unroll
    for (int x = 0; x < 2 * MB; ++x) tra[x] = tr_addr(tr_lane, x);
    // block 0 up to its scores, the fragments of block 1 (tiles 0 and 1 have landed)
#pragma unroll
    for (int ks = 0; ks < KS; ++ks) { mfma32_settle<AGPR>(qreg[ks]); mfma32_settle<AGPR>(doreg[ks]); }
#pragma unroll
    for (int ks = 0; ks < KS; ++ks) { row_frag(rm_addr(rm_lane, ks), 0, ks); row_frag(rm_addr(rm_lane, ks), 0, KS + ks); }
#pragma unroll
    for (int i = 0; i < kA; ++i) start(s0, d0, i);
    mfma32_fixed_done(s0);
    mfma32_fixed_done(d0);
#pragma unroll
    for (int ks = 0; ks < KS; ++ks) { row_frag(rm_addr(rm_lane, ks), 1, ks); row_frag(rm_addr(rm_lane, ks), 1, KS + ks); }
    // the tile requested in an iteration (past the last one that one again)
    int req = min(R.startup_tiles, n_kt - 1);
    const char* k_it = kbase + (int64_t)req * kBK * kstep;
    const char* v_it = vbase + (int64_t)req * kBK * vstep;
    TileLaneOff<D> lane_off = tile_lane_offsets<D>(kstep, vstep, min(p.Sk - req * kBK, kBK), src.x, src.y);
    int stage = 0, jt = 0;
    uint32_t req_dst = wave_dst + R.startup_tiles * kStageBytes;
    // loads of the first and second half of a tile, in the second halves of its two steps: every kEvery slots
    constexpr int kLoads = 2 * Z::kPasses, kEvery = 2 * kB / kLoads, kPerStep = kLoads / 2;
    auto load = [&](int k) { issue_tile_load<D>(k, k_it, v_it, lane_off, req_dst); };
    auto request = [&](int first) {  // outside the steps
#pragma unroll
      for (int k = 0; k < kPerStep; ++k) load(first + k);
    };
    auto end_tile = [&]() {
      wait_vmcnt<ring::loads_kept_after_iteration(R, true)>();
      // a bare barrier: every read of this tile has returned (the products used it), and the next tile's fragments that
      // are still on their way come from a stage that the next iteration does not refill either
      asm volatile("" ::: "memory");
      __builtin_amdgcn_s_barrier();
      asm volatile("" ::: "memory");
      stage = stage == kStages - 1 ? 0 : stage + 1;
      req_dst += kStageBytes;
      if (req_dst >= lds0 + kStages * kStageBytes) req_dst -= kStages * kStageBytes;
      if (req + 1 < n_kt) {
        ++req;
        k_it += kBK * kstep;
        v_it += (int64_t)kBK * vstep;
        if (p.Sk - req * kBK < kBK) lane_off = tile_lane_offsets<D>(kstep, vstep, p.Sk - req * kBK, src.x, src.y);
      }
    };
    auto first_step = [&](auto masked_c) {
      step(masked_c, s0, d0, s1, d1, 0, kBK * jt,
           [&](int slot) { const int j = slot - kA; if (j >= 0 && j % kEvery == kEvery - 1) load(j / kEvery); }, [](int) {});
    };
    auto second_step = [&](auto masked_c) {
      uint32_t rm_next = 0, tr_next = 0;
      step(masked_c, s1, d1, s0, d0, 1, kBK * jt + 32,
           [&](int slot) { const int j = slot - kA; if (j >= 0 && j % kEvery == kEvery - 1) load(kPerStep + j / kEvery); },
           [&](int slot) {  // the next iteration's addresses, each behind its last use in this one
             const int j = slot - kA;
             if (j == 0) {
               tr_next = tr_lane + (stage == kStages - 1 ? 0 : stage + 1) * kStageBytes;
               rm_next = rm_lane + (stage >= kStages - 2 ? stage + 2 - kStages : stage + 2) * kStageBytes;
             }
             if (j >= 0) tra[j] = tr_addr(tr_next, j);
#pragma unroll
             for (int ks = 0; ks < KS; ++ks)
               if (j == (ks < KS / 2 ? ks + 1 : ks < KS - 2 ? KS - 3 : ks)) rma[ks] = rm_addr(rm_next, ks);
           });
    };
    for (; jt < n_a; ++jt) {
      first_step(IC<0>{});
      second_step(IC<0>{});
      end_tile();
    }
    for (; 2 * jt + 1 < n_act; ++jt) {
      first_step(IC<1>{});
      second_step(IC<1>{});
      end_tile();
    }
    for (; jt < n_kt; ++jt) {  // tiles of which this wave needs one block, then none
      if (2 * jt < n_act) first_step(IC<2>{});
      else request(0);
      request(kPerStep);
      end_tile();
    }
#pragma unroll
    for (int mb = 0; mb < MB; ++mb) mfma32_acc_done<AGPR>(acc[mb]);
    static_assert(R.always_requests, "no branch around the loads of an iteration");
    wait_vmcnt<0>();  // the last tile, requested once more, has left the stages that the epilogue uses
    __syncthreads();
  } else {
    auto request_rowmajor = [&](uint32_t rm, int kb) {  // kb compile-time at every call site
#pragma unroll
      for (int ks = 0; ks < KS; ++ks) {
        kf[ks] = swz_frag_rm<D>(rm, kb, ks);
        vf[ks] = swz_frag_rm<D>(rm + Z::kTileBytes, kb, ks);
      }
    };
    // one 32-key block: tr = lane address inside the block's stage; `more`: a block follows, its row-major
    // fragments start at next_rm
    // MASKED is compile-time so that a whole block is one straight-line scheduling region
    auto step = [&](auto masked_c, uint32_t tr, int kb, int jb, uint32_t next_rm, int next_kb) {
      constexpr bool MASKED = decltype(masked_c)::value != 0;
      // head_dim 128 (64-row workgroups here) runs one wave per SIMD with all 256 ordinary registers in use: left to itself the compiler requests
      // each LDS fragment one MFMA ahead of its use and the wave stalls on LDS latency before most MFMAs.  Asking for
      // the block as 24 groups of (1 MFMA, 2 LDS reads, 2 vector instructions) keeps two requests ahead: -6 % on this
      // kernel (neighbouring group shapes are 2-10 % slower; at head_dim 64, two waves per SIMD, none changes anything).
      if constexpr (D == 128) {
#pragma unroll
        for (int i = 0; i < 3 * KS; ++i) {
          __builtin_amdgcn_sched_group_barrier(0x008, 1, 0);  // MFMA
          __builtin_amdgcn_sched_group_barrier(0x100, 2, 0);  // LDS read
          __builtin_amdgcn_sched_group_barrier(0x002, 2, 0);  // VALU
        }
      }
      f32x16 s = c_lse, dpv = c_del;
      // the S chain first, then the dP chain: exp2 of the finished scores runs behind the dP MFMAs
#pragma unroll
      for (int ks = 0; ks < KS; ++ks) s = mfma32(kf[ks], qreg[ks], s);
#pragma unroll
      for (int ks = 0; ks < KS; ++ks) dpv = mfma32(vf[ks], doreg[ks], dpv);
      bf16x8 kT[MB][2];
#pragma unroll
      for (int mb = 0; mb < MB; ++mb) {
        kT[mb][0] = swz_frag_tr<D>(tr, mb, 2 * kb);
        kT[mb][1] = swz_frag_tr<D>(tr, mb, 2 * kb + 1);
      }
      if (MASKED) {  // block touches the diagonal or the end of the keys
        // register r holds key jb + 4hh + c_r, c_r = 8(r/4) + r%4: masked iff c_r > qlim - jb - 4hh
        const int t = qlim - jb - 4 * hh;
#pragma unroll
        for (int r = 0; r < 16; ++r)
          if (8 * (r >> 2) + (r & 3) > t) s[r] = -INFINITY;
      }
#pragma unroll
      for (int r = 0; r < 16; ++r) s[r] = fast_exp2(s[r]) * dpv[r];
      const bf16x8 ds0 = pack_c_half(s, 0), ds1 = pack_c_half(s, 1);
      request_rowmajor(next_rm, next_kb);  // unconditional: past the last block the fragments are simply unused
#pragma unroll
      for (int mb = 0; mb < MB; ++mb) {
        acc[mb] = mfma32(kT[mb][0], ds0, acc[mb]);
        acc[mb] = mfma32(kT[mb][1], ds1, acc[mb]);
      }
    };

    if (n_act > 0) request_rowmajor(rm_lane, 0);
    int stage = 0, jt = 0;
    for (; jt < n_a; ++jt) {
      const int nstage = stage == kStages - 1 ? 0 : stage + 1;
      const uint32_t rm = rm_lane + stage * kStageBytes, tr = tr_lane + stage * kStageBytes;
      if constexpr (PARTS == 1) {
        step(IC<0>{}, tr, 0, 64 * jt, rm, 1);
        step(IC<0>{}, tr, 1, 64 * jt + 32, rm_lane + nstage * kStageBytes, 0);
      } else {
        step(IC<0>{}, tr, 0, 64 * jt + 32 * part, rm_lane + nstage * kStageBytes, 0);
      }
      // stage (jt+3) % 4 == (jt-1) % 4 was last read in the previous iteration: refill it, then make sure
      // this wave's part of tile jt+2 (needed from the next iteration's prefetch on) has landed
      if (jt + R.issue_ahead < n_kt) { issue_tile(jt + R.issue_ahead); wait_vmcnt<ring::loads_kept_after_iteration(R, true)>(); } else wait_vmcnt<ring::loads_kept_after_iteration(R, false)>();
      __syncthreads();
      stage = nstage;
    }
    for (; jt < n_kt; ++jt) {
      const int nstage = stage == kStages - 1 ? 0 : stage + 1;
      const uint32_t rm = rm_lane + stage * kStageBytes, tr = tr_lane + stage * kStageBytes;
      if constexpr (PARTS == 1) {
        if (2 * jt < n_act) step(IC<1>{}, tr, 0, 64 * jt, rm, 1);
        if (2 * jt + 1 < n_act) step(IC<1>{}, tr, 1, 64 * jt + 32, rm_lane + nstage * kStageBytes, 0);
      } else {
        if (2 * jt + part < n_act) step(IC<1>{}, tr, 0, 64 * jt + 32 * part, rm_lane + nstage * kStageBytes, 0);
      }
      if (jt + R.issue_ahead < n_kt) { issue_tile(jt + R.issue_ahead); wait_vmcnt<ring::loads_kept_after_iteration(R, true)>(); } else wait_vmcnt<ring::loads_kept_after_iteration(R, false)>();
      __syncthreads();
      stage = nstage;
    }
  }

  // ---- epilogue.  First what the dK/dV kernel reads of this row: Qhat, -delta, -lse2 (and dgate).  A gate factor
  // f > 0 reaches that kernel through the two statistics and it streams the caller's dO as it is: with
  // P' = f P = exp2(S - lse2 + log2 f) it holds dV' = P'^T dO and dS = P (f dP - delta) = P' (dP - delta / f).  A
  // factor that underflowed switches the row off (P' = 0).  Only a gate scale <= 0 needs the gated copy of dO.
  // With a rotary embedding the table rows come in once more, into the idle ring (every wave has passed the last
  // iteration's barrier), now for the accumulators' layout; the second barrier keeps the scale-gradient staging
  // below, which reuses the ring, behind every wave's reads.
  // PARTS == 2: part 1 leaves its T^T in the idle stage 2 (one slot per wave, 16 bytes per lane and access: conflict-free)
  // and is done but for the column sums; part 0 adds it to its own.
  char* const slot = lds + R.merge_stage_first * kStageBytes + row_wave * (MB * 4096) + lane * 16;
  static_assert(PARTS == 1 || (kRowWaves * MB * 4096 <= R.merge_stages * kStageBytes && BQ * kRedStride * 4 <= R.scratch_stages * kStageBytes &&
                               R.scratch_stages <= R.merge_stage_first), "slots behind the dg staging area");
  if constexpr (PARTS == 2) {
    if (part == 1) {
#pragma unroll
      for (int mb = 0; mb < MB; ++mb)
#pragma unroll
        for (int c = 0; c < 4; ++c)
          *reinterpret_cast<f32x4*>(slot + (4 * mb + c) * 1024) = f32x4{acc[mb][4 * c], acc[mb][4 * c + 1], acc[mb][4 * c + 2], acc[mb][4 * c + 3]};
    }
    if constexpr (!ROPE) __syncthreads();
  }
  RopeCt<MB> rope_ct;
  if constexpr (ROPE) {
    constexpr uint32_t kSinAt = PARTS == 1 ? kStageBytes : kPair;
    issue_rope_rows(0, kSinAt);
    wait_vmcnt<0>();
    __syncthreads();
    rope_ct = rope_ct_from_lds<MB>(row16, row16 + kSinAt, hh);
    __syncthreads();
  }
  float* red = reinterpret_cast<float*>(lds);
  if (PARTS == 1 || part == 0) {
    if constexpr (PARTS == 2) {
#pragma unroll
      for (int mb = 0; mb < MB; ++mb)
#pragma unroll
        for (int c = 0; c < 4; ++c) {
          const f32x4 t = *reinterpret_cast<const f32x4*>(slot + (4 * mb + c) * 1024);
#pragma unroll
          for (int i = 0; i < 4; ++i) acc[mb][4 * c + i] += t[i];
        }
    }
    if (live) {
#pragma unroll
      for (int ks = 0; ks < KS; ++ks) {
        *reinterpret_cast<bf16x8*>(a.qhat + head_row * D + (int64_t)row_c * D + 16 * ks + 8 * hh) = qreg[ks];
        if (a.do_eff) *reinterpret_cast<bf16x8*>(reinterpret_cast<uint16_t*>(a.do_eff) + head_row * D + (int64_t)row_c * D + 16 * ks + 8 * hh) = doreg[ks];
      }
      if (hh == 0) {
        float stat_d = -delta, stat_l = nlse2;
        if (p.gate.ptr && !a.do_eff) {
          const bool on = gfac > kGateFactorFloor;
          stat_l = on ? nlse2 + __log2f(gfac) : -INFINITY;
          stat_d = on ? -delta / gfac : 0.f;
        }
        (a.delta + head_row)[row_c] = stat_d;
        (a.nlse2 + head_row)[row_c] = stat_l;
        if (p.gate.ptr)
          reinterpret_cast<uint16_t*>(p.dgate.ptr)[(int64_t)b * p.dgate.stride_b + (int64_t)row * p.dgate.stride_s + (int64_t)h * p.dgate.stride_h] = f32_to_bf16(dgate_row);
      }
    }
    // acc = T^T: lane = query, registers = head-dim entries.
    float dot = 0.f;
    // q in the C-tile layout (rotated like the operand was), then dq = a (u - (a^2/D)(u.q) q) in the rotated frame
    // and back through the transpose of the rotation
    float qv[MB][16];
#pragma unroll
    for (int mb = 0; mb < MB; ++mb) unpack_ct_block(qct[mb], qv[mb]);
    const float aq = live ? alpha : 0.f;  // padding rows add nothing to the scale gradient
    if (ROPE) rope_ct_apply<MB, false>(qv, rope_ct);
#pragma unroll
    for (int mb = 0; mb < MB; ++mb) {
#pragma unroll
      for (int c = 0; c < 4; ++c) {
        const int d0 = 32 * mb + 8 * c + 4 * hh;
        const float4 g4 = *reinterpret_cast<const float4*>(gsm + d0);
        const float gv[4] = {g4.x, g4.y, g4.z, g4.w};
        float dgc[4];
#pragma unroll
        for (int i = 0; i < 4; ++i) {
          const int r = 4 * c + i;
          const float t = acc[mb][r] * p.sm_scale;                 // sm_scale * T
          dgc[i] = t * aq * qv[mb][r];                             // dg contribution of this row
          acc[mb][r] = t * gv[i];                                  // u = dL/d(a q)
          dot += acc[mb][r] * qv[mb][r];
        }
        *reinterpret_cast<float4*>(red + (row_wave * 32 + ln) * kRedStride + d0) = make_float4(dgc[0], dgc[1], dgc[2], dgc[3]);
      }
    }
    dot = half_sum(dot);
    const float a3 = norm_grad_coef(p, alpha, 1.0f / D) * dot;
    uint16_t* op = row_ptr_mut<uint16_t>(p.dq, b, h, row_c);
    float val[MB][16];
#pragma unroll
    for (int mb = 0; mb < MB; ++mb)
#pragma unroll
      for (int r = 0; r < 16; ++r) val[mb][r] = alpha * acc[mb][r] - a3 * qv[mb][r];
    if (ROPE) rope_ct_apply<MB, true>(val, rope_ct);
#pragma unroll
    for (int mb = 0; mb < MB; ++mb) store_ct_block(op, mb, hh, live, val[mb]);
  }
  // workgroup partial of dg: column sums over the BQ (wave, lane%32) rows, in two levels so that all
  // 256 threads share the LDS reads (fixed order: deterministic)
  __syncthreads();
  {
    const int cg = tid % kColGroups, rg = tid / kColGroups;
    float4 t = make_float4(0.f, 0.f, 0.f, 0.f);
#pragma unroll
    for (int x = 0; x < kRowsPerGroup; ++x) {
      const float4 v = *reinterpret_cast<const float4*>(red + (rg * kRowsPerGroup + x) * kRedStride + 4 * cg);
      t.x += v.x; t.y += v.y; t.z += v.z; t.w += v.w;
    }
    *reinterpret_cast<float4*>(red4 + rg * D + 4 * cg) = t;
  }
  __syncthreads();
  if (tid < D) {
    float t = 0.f;
#pragma unroll
    for (int x = 0; x < kRowGroups; ++x) t += red4[x * D + tid];
    a.dg_part[(int64_t)blockIdx.x * D + tid] = t;
  }
}

// ============================================================================================ dK, dV
// Same pipeline with the roles swapped: the streamed tiles are Qhat / dO (64 queries of one head), the
// blocks are 32 queries, and B(n) starts from the two row statistics of the block, read from LDS
// straight into the accumulators of S and dP.  PARTS: see dkdv_parts(); with 2 a wave computes one block of every tile
// and the two waves of a key block add up their accumulators through LDS behind the loop.
// PIPE (PARTS == 1): see dkdv_pipelined().
template <int D, bool ROPE, int PARTS, bool PIPE>
__global__ __launch_bounds__(kThreadsM, D == 64 ? 2 : 1) void bwd_dkdv_bf16_kernel(KArgs a) {
  using Z = Swz<D>;
  static_assert(PARTS == 1 || (PARTS == 2 && !PIPE), "a tile has two 32-query blocks");
  constexpr int BKV = kBwdRows / PARTS;
  constexpr int kKeyWaves = 4 / PARTS;  // waves side by side along the keys
  constexpr int KS = D / 16;
  constexpr int MB = D / 32;
  constexpr int kStageBytes = 2 * Z::kTileBytes;
  constexpr ring::Protocol R = PARTS == 1 ? ring::dkdv(Z::kPasses, PIPE) : ring::dkdv_parts(Z::kPasses);  // the pipeline's numbers: ring_protocol.hpp
  static_assert(ring::well_formed(R) && R.stages == kStages && R.row_stages == 2 && !R.wait_before_loop && !R.issue_at_top, "tile pipeline");
  static_assert(R.early_tiles >= ring::kTilesNeededAtLoopStart, "the loop is entered without a further wait");
  static_assert(R.loads_per_tile == 2 * Z::kPasses + 1, "per wave: the two tiles plus one row-statistics load");
  const segpt_attn_params& p = a.p;
  __shared__ __attribute__((aligned(1024))) char lds[kStages * kStageBytes];
  __shared__ __attribute__((aligned(256))) float ldl[kStages * 128];  // per stage: [0,64) -lse2, [64,128) -delta
  __shared__ float red[8];

  const int tid = threadIdx.x, lane = tid & 63;
  const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);  // wave-uniform: everything derived from it stays scalar
  const int ln = lane & 31, hh = lane >> 5;
  const int rep = __builtin_amdgcn_readfirstlane(p.H / p.Hkv);  // divided in vector registers
  const int n_kvt = (p.Sk + BKV - 1) / BKV;
  // Workgroup 0 is an extra one: dispatched first, it only folds the dQ kernel's per-workgroup partials of the
  // scale-vector gradient (complete: that kernel ran before this one on the stream) while the others compute.
  if (blockIdx.x == 0) {
    float* red = reinterpret_cast<float*>(lds);
    reduce_scale_grad<kThreadsM>(a, tid, red, red + kThreadsM);
    return;
  }
  const int bid = blockIdx.x - 1;  // still a fixed rotation of the hardware's round-robin over the XCDs
  WgCoord wg = decode_wg(bid, n_kvt, p.B, p.Hkv, 1, dkdv_pinned(p));
  if (!wg.valid) {  // idle padding workgroup: its (dc1, dc2) partial must still read as zero
    if (tid < 2) a.dcoef_part[(int64_t)bid * 2 + tid] = 0.f;
    return;
  }
  wg.tile = __builtin_amdgcn_readfirstlane(n_kvt - 1 - wg.tile);  // early key tiles see the most queries: issue them first
  const int b = __builtin_amdgcn_readfirstlane(wg.b), g = __builtin_amdgcn_readfirstlane(wg.g);
  const int k0 = wg.tile * BKV;
  const int key_wave = PARTS == 1 ? wave : wave % kKeyWaves, part = PARTS == 1 ? 0 : wave / kKeyWaves;
  const int kw0 = k0 + key_wave * 32;
  const int key = kw0 + ln;
  const int key_c = min(key, p.Sk - 1);

  const int n_qt = (p.Sq + kBK - 1) / kBK;
  int qt_start = 0;
  if (p.causal) qt_start = min(max(0, k0 - p.q_start) / kBK, n_qt);
  const int n_vis = n_qt - qt_start;  // visible query tiles per head
  const int n_it = __builtin_amdgcn_readfirstlane(n_vis * rep);  // streamed tiles in total

  // ---- staging of one (head, query tile): Qhat and dO tiles plus the two row statistics, all by direct
  // global->LDS loads.  Every wave issues the same number of loads (waves 2/3 repeat the statistics load
  // of waves 0/1) so that one immediate vmcnt fits all.
  const uint32_t lds0 = lds_addr_of(lds), ldl0 = lds_addr_of(ldl);
  const int2 src = swz_src<D>(lane, wave);
  const bool do_contig = a.do_eff != nullptr;
  const float* const stat_arr = (wave & 1) ? a.delta : a.nlse2;
  const uint32_t dstep = do_contig ? (uint32_t)D * 2 : (uint32_t)p.d_o.stride_s * 2;
  const TileLaneOff<D> full_tile = tile_lane_offsets<D>(D * 2, dstep, kBK, src.x, src.y);
  // The stream of (query tile, head) pairs is walked by running pointers kept beside the compute loop's own counters
  // (three tiles ahead of it): per tile a few scalar additions.
  // PIPE: from the last tile down, every head of the group at a tile before the next tile.  All workgroups of a
  // (batch, kv head) pair start at the same tile and stay together, so that a tile comes into the XCD's L2 once for all of them.
  // Head by head and upwards from the diagonal every workgroup was somewhere else: L2 misses per launch (128-byte lines),
  // 4 x 16 / 4 heads, 4096 tokens, head_dim 128 9.8 M -> 4.0 M, 2 x 18 / 6 heads, 8192 tokens, head_dim 64 10.7 M -> 3.9 M.
  // Without, head by head and upwards: these launches' streams are short and fit the L2 anyway, and in step their workgroups
  // only queue for the same lines (8 x 18 / 6 heads, 999 tokens: the whole step 177.3 us, in step 178.5).
  constexpr bool kInStep = PIPE;
  int iss_h = 0, iss_t = 0, iss_stage = 0, issued = 0;
  const int i_first = kInStep ? (n_qt - 1) * kBK : qt_start * kBK;  // first query of the stream's first tile
  const int64_t row_first = ((int64_t)b * p.H + g * rep) * p.Sq + i_first;
  const int64_t q_head = (int64_t)p.Sq * D * 2, d_head = do_contig ? q_head : (int64_t)p.d_o.stride_h * 2;
  const char* q_it = reinterpret_cast<const char*>(a.qhat + row_first * D);
  const char* d_it = do_contig ? reinterpret_cast<const char*>(reinterpret_cast<const uint16_t*>(a.do_eff) + row_first * D)
                               : reinterpret_cast<const char*>(row_ptr<uint16_t>(p.d_o, b, g * rep, i_first));
  const float* s_it = stat_arr + row_first;
  int left_it = p.Sq - i_first;
  auto move = [&](int tiles, int heads) {
    const int rows = tiles * kBK;
    q_it += heads * q_head + (int64_t)rows * D * 2;
    d_it += heads * d_head + (int64_t)rows * dstep;
    s_it += heads * p.Sq + rows;
    left_it -= rows;
  };
  auto advance = [&]() {
    if constexpr (kInStep) {
      if (++iss_h == rep) { iss_h = 0; move(-1, 1 - rep); } else move(0, 1);
    } else {
      if (++iss_t == n_vis) { iss_t = 0; move(1 - n_vis, 1); } else move(1, 0);
    }
  };
  const uint32_t lane4 = lane * 4;
  auto issue_next = [&]() {
    const uint32_t dst = lds0 + iss_stage * kStageBytes + wave * 1024;
    const uint32_t sdst = ldl0 + (iss_stage * 128 + (wave & 1) * 64) * 4;
    if (left_it >= kBK) {
      issue_tile_pair<D>(q_it, d_it, full_tile, dst);
      gload_lds4_so(s_it, lane4, sdst);
    } else {
      issue_tile_pair<D>(q_it, d_it, tile_lane_offsets<D>(D * 2, dstep, left_it, src.x, src.y), dst);
      gload_lds4_so(s_it, (uint32_t)min(lane, left_it - 1) * 4, sdst);
    }
    iss_stage = iss_stage == kStages - 1 ? 0 : iss_stage + 1;
    if (++issued < n_it) advance();
  };

  // ---- start-up: streamed tiles 0 and 1 into stages 0 and 1, and with them the workgroup's 128 Khat and V' rows
  // as tiles into stages 2 and 3 (whole cache lines by direct loads instead of 16 bytes per lane and row; the
  // row-major fragment read of a tile is the B-operand layout): one memory round trip.  Once the rows sit in
  // registers, tile 2 is requested into stage 2 and the ring turns as usual (every iteration needs its own tile and
  // the next one landed, and leaves one more in flight).
#pragma unroll
  for (int t = 0; t < R.early_tiles; ++t)
    if (t < n_it) issue_next();
  constexpr int kRowStage = R.row_stage_first;  // Khat block in stage kRowStage, V' block in the next
  {
    const int rows_left = min(p.Sk - k0, BKV);
    const int64_t krow = ((int64_t)b * p.Hkv + g) * p.Sk + k0;
    const char* kb = reinterpret_cast<const char*>(a.khat + krow * D);
    const char* vb = a.vmix ? reinterpret_cast<const char*>(a.vmix + krow * D) : reinterpret_cast<const char*>(row_ptr<uint16_t>(p.v, b, g, k0));
    const uint32_t vstep = a.vmix ? (uint32_t)D * 2 : (uint32_t)p.v.stride_s * 2;
    const uint32_t wave_dst = lds0 + wave * 1024;
    if constexpr (PARTS == 1) {
      issue_tile_pair<D>(kb, kb, rowblock_lane_offsets<D>(D * 2, 0, rows_left, src.x, src.y), wave_dst + kRowStage * kStageBytes);
      issue_tile_pair<D>(vb, vb, rowblock_lane_offsets<D>(vstep, 0, rows_left, src.x, src.y), wave_dst + (kRowStage + 1) * kStageBytes);
    } else {  // 64 rows each: the two tiles of one stage
      issue_tile_pair<D>(kb, vb, tile_lane_offsets<D>(D * 2, vstep, rows_left, src.x, src.y), wave_dst + kRowStage * kStageBytes);
    }
  }
  wait_vmcnt<0>();
  __syncthreads();
  // stationary B operands: Khat and V' rows of this lane's key (rows 32*key_wave .. +31 of the block)
  bf16x8 kreg[KS], vreg[KS];
  {
    const uint32_t rm = lds0 + kRowStage * kStageBytes + (key_wave >> 1) * Z::kTileBytes + swz_off_rm<D>(lane);
    const int rb = key_wave & 1;
    constexpr int kVRows = PARTS == 1 ? kStageBytes : Z::kTileBytes;  // where the V' rows lie behind the Khat rows
#pragma unroll
    for (int ks = 0; ks < KS; ++ks) {
      kreg[ks] = swz_frag_rm<D>(rm, rb, ks);
      vreg[ks] = swz_frag_rm<D>(rm + kVRows, rb, ks);
    }
  }
  __syncthreads();  // the borrowed stages are free again
#pragma unroll
  for (int t = R.early_tiles; t < R.startup_tiles; ++t)
    if (t < n_it) issue_next();
  f32x16 dvacc[MB], dkacc[MB];
#pragma unroll
  for (int mb = 0; mb < MB; ++mb) { dvacc[mb] = splat16(0.f); dkacc[mb] = splat16(0.f); }

  // PARTS == 2: this wave's block of every tile is number `part` (a multiple of 4 KB further: the XOR terms stay below)
  const uint32_t rm_lane = lds0 + swz_off_rm<D>(lane) + part * 32 * Z::kRB;
  const uint32_t tr_lane = lds0 + swz_off_tr<D>(lane) + part * 32 * Z::kRB;
  const uint32_t st_lane = ldl0 + 16 * hh + part * 32 * 4;

  bf16x8 qf[KS], df[KS];
  // The visible query tiles t = 0 .. n_vis-1 (first query (qt_start + t) * 64) fall into runs for this wave: [0, t_diag)
  // touch the causal diagonal (those before t_full lie inside Sq and need the diagonal test only), [t_diag, t_end) need
  // no mask, [t_end, n_vis) run past Sq.  Each run is its own loop so that a loop body holds one variant of the block
  // (whole-block scheduling regions, no accumulator copies at joins).
  int t_diag = 0;
  if (p.causal) t_diag = min(max((max(kw0 + 31 - p.q_start, 0) + kBK - 1) / kBK - qt_start, 0), n_vis);
  const int t_full = min(max(p.Sq / kBK - qt_start, 0), n_vis);  // tiles whose 64 queries all exist
  const int t_end = max(t_full, t_diag);
  if constexpr (PIPE) {
    // A software pipeline over 32-query blocks, laid out instruction by instruction: step n computes the scores and dP of
    // block n + 1 (first half: kA matrix instructions) while the vector unit turns those of block n into P and dS, then
    // adds block n to dV and dK (second half: kB) while the row-major fragments and row statistics of block n + 2 come in.
    // A slot is one matrix instruction and what fits beside it, closed by a scheduling barrier, so that the source's order is
    // the kernel's.  What a slot holds (one wave per SIMD, cycles): a matrix instruction runs for 32 and keeps the vector
    // port for 16 of them; behind it a plain vector instruction takes 4, an exponential 8, an LDS read 8 (for free in
    // those 16), a direct load 13.  Left to the compiler, the products of a block ran first and its exponentials next.
    // The accumulators and the stationary rows live in accumulation registers, scores and dP in ordinary ones; a kernel
    // of more than 256 registers gets one form for all matrix instructions from the compiler, hence the inline assembly,
    // whose wait states tests/test_mfma_hazards.py checks on the built code.
    // dK/dV, us: head_dim 128, 4 x 16 / 4 heads, 4096 tokens 543 -> 451 (1159 k -> 741 k cycles, matrix pipe 46 -> 71 % busy; the
    // card holds its power, so the clock gives part of it back, 2.13 -> 1.64 GHz); head_dim 64, 2 x 18 / 6 heads, 8192 tokens 599 ->
    // 556 (54 -> 67 %), 8 x 2048 161 -> 156 (48 -> 55 %).
    constexpr int kA = 2 * KS, kB = 4 * MB;
    // i-th product of the first half: k-step of S (0 .. KS-1) or KS + that of dP.  S leads, so that the statistics from which
    // dP starts, requested last, have time.
    constexpr int kOrder64[] = {0, 1, 4, 2, 5, 3, 6, 7}, kOrder128[] = {0, 1, 2, 8, 3, 9, 4, 10, 5, 11, 6, 12, 7, 13, 14, 15};
    auto order = [&](int i) { return D == 64 ? kOrder64[i & 7] : kOrder128[i]; };
    f32x16 s0, d0, s1, d1;  // scores and dP of two consecutive blocks
    uint32_t rm_next = 0, st_next = 0;        // the next tile's row-major fragments and statistics
    uint32_t rma[KS], tra[2 * MB];            // ... its fragments by k-step, and this tile's transposed ones by column block
    auto load_stat = [&](f32x16& s, f32x16& d, uint32_t st, int qb, int c) {  // a quarter of -lse2 (c < 4) or -delta
      const f32x4 v = lds_read_f4(st + ((c & 4 ? 64 : 0) + 32 * qb + 8 * (c & 3)) * 4);
#pragma unroll
      for (int i = 0; i < 4; ++i) (c & 4 ? d : s)[4 * (c & 3) + i] = v[i];
    };
    // (s, d): block n, whose first query is ib, number qb of its tile; (sn, dn): block n + 1.  mem and alu: what else
    // the slots hold, beside the LDS reads and beside the vector instructions.  The mask variant is compile-time: 0 none, 1 causal
    // diagonal only (every query of the block exists), 2 diagonal and / or end of the queries.
    auto step = [&](auto masked_c, f32x16& s, f32x16& d, f32x16& sn, f32x16& dn, int qb, int ib, auto mem, auto alu) {
      constexpr int MASK = decltype(masked_c)::value;
      // register r holds query ib + 4hh + c_r with c_r = 8(r/4) + r%4 a compile-time constant.
      // masked iff key > query + q_start  <=>  c_r < key - q_start - ib - 4hh,   or query >= Sq
      const int t = p.causal ? key - p.q_start - ib - 4 * hh : -1;
      const int u = p.Sq - ib - 4 * hh;
      u32x4 pw[2], dw[2];  // P and dS as operands, in halves of 16 queries
      bf16x8 dT[MB][2], qT[MB][2];
      auto v_exp = [&](int r) {
        const int c = 8 * (r >> 2) + (r & 3);
        if (MASK == 1 ? c < t : MASK == 2 && (c < t || c >= u)) s[r] = -INFINITY;
        s[r] = fast_exp2(s[r]);
      };
      auto v_mul = [&](int r, int n) {
        for (int i = r; i < r + n; ++i) d[i] *= s[i];
      };
      auto v_p = [&](int j, int n) {
        for (int i = j; i < j + n; ++i) pw[i >> 2][i & 3] = pack_bf16x2(s[2 * i], s[2 * i + 1]);
      };
      auto v_ds = [&](int j, int n) {
        for (int i = j; i < j + n; ++i) dw[i >> 2][i & 3] = pack_bf16x2(d[2 * i], d[2 * i + 1]);
      };
#pragma unroll
      for (int i = 0; i < kA; ++i) {
        const int o = order(i);
        if (o < KS) mfma32_fixed(sn, qf[o], kreg[o]);
        else mfma32_fixed(dn, df[o - KS], vreg[o - KS]);
        const int half = i / (2 * MB), mb = (i % (2 * MB)) >> 1;
        (i & 1 ? qT : dT)[mb][half] = frag_tr_at<D>(tra[2 * mb], tra[2 * mb + 1], 2 * qb + half, i & 1 ? 0 : Z::kTileBytes);
        mem(i);
        __builtin_amdgcn_sched_barrier(0);
        if constexpr (D == 128) {
          v_exp(i);
          if (i >= 1 && i <= 8) v_mul(i - 1, 1);
          if (i >= 9 && i <= 12) v_p(i - 9, 1);
          if (i >= 13) v_ds(i - 13, i == 15 ? 2 : 1);
        } else {
          v_exp(2 * i);
          v_exp(2 * i + 1);
          if (i >= 1 && i <= 4) v_mul(2 * i - 2, 2);
          if (i == 5 || i == 6) v_p(2 * i - 10, 2);
          if (i == 7) v_ds(0, 4);
        }
        alu(i);
        __builtin_amdgcn_sched_barrier(0);
      }
#pragma unroll
      for (int j = 0; j < kB; ++j) {
        const int half = j / (2 * MB), mb = (j % (2 * MB)) >> 1;
        if (j & 1) mfma32_acc(dkacc[mb], qT[mb][half], as_bf16x8(dw[half]));
        else mfma32_acc(dvacc[mb], dT[mb][half], as_bf16x8(pw[half]));
        const int o = order(j);
        (o < KS ? qf : df)[o % KS] = as_bf16x8(lds_read16(rma[o % KS] + (o < KS ? 0 : Z::kTileBytes) + qb * 32 * Z::kRB));
        if (D == 128 && j >= 6 && j < 14) load_stat(s, d, st_next, qb, j - 6);
        if (D == 64 && j >= 4) {
          load_stat(s, d, st_next, qb, 2 * (j - 4));
          load_stat(s, d, st_next, qb, 2 * (j - 4) + 1);
        }
        mem(kA + j);
        __builtin_amdgcn_sched_barrier(0);
        if constexpr (D == 128) {
          if (j < 2) v_mul(8 + 3 * j, 3);
          if (j == 2) { v_mul(14, 2); v_p(4, 1); }
          if (j == 3) v_p(5, 3);
          if (j == 4) v_ds(4, 3);
          if (j == 5) v_ds(7, 1);
        } else {
          if (j < 2) v_mul(8 + 4 * j, 4);
          if (j == 2) v_p(4, 4);
          if (j == 3) v_ds(4, 4);
        }
        alu(kA + j);
        __builtin_amdgcn_sched_barrier(0);
      }
    };
    auto tr_addr = [&](uint32_t tr, int x) { return tr ^ (uint32_t)(((x >> 1) << 6) ^ (x & 1 ? Z::kHiXor : 0)); };
#pragma unroll
    for (int x = 0; x < 2 * MB; ++x) tra[x] = tr_addr(tr_lane, x);
    if (n_it > 0) {  // tiles 0 and 1 have landed (first wait above): block 0 up to its scores, the fragments of block 1
#pragma unroll
      for (int qb = 0; qb < 2; ++qb) {
#pragma unroll
        for (int ks = 0; ks < KS; ++ks) {
          qf[ks] = swz_frag_rm<D>(rm_lane, qb, ks);
          df[ks] = swz_frag_rm<D>(rm_lane + Z::kTileBytes, qb, ks);
        }
#pragma unroll
        for (int c = 0; c < 8; ++c) load_stat(qb ? s1 : s0, qb ? d1 : d0, st_lane, qb, c);
        if (qb == 0) {
#pragma unroll
          for (int ks = 0; ks < KS; ++ks) {
            mfma32_fixed(s0, qf[ks], kreg[ks]);
            mfma32_fixed(d0, df[ks], vreg[ks]);
          }
          mfma32_fixed_done(s0);
          mfma32_fixed_done(d0);
        }
      }
    }
    // the tile requested in an iteration: its rows' lane offsets, cut off at the last query, and where the stream goes on
    const uint32_t q_row = (uint32_t)src.x * D * 2, d_row = (uint32_t)src.x * dstep;
    const int64_t q_wrap = -((rep - 1) * q_head + kBK * D * 2), d_wrap = -((rep - 1) * d_head + (int64_t)kBK * dstep);
    const int s_wrap = -((rep - 1) * p.Sq + kBK);
    constexpr int kLoads = 2 * Z::kPasses;
    // slots of the second halves that hold load k (first step: k < kFirst) and, one slot before, its offset
    constexpr int kFirst = D == 128 ? 5 : 3, kAt0 = D == 128 ? 7 : 4, kAt1 = D == 128 ? 6 : 4, kEvery = D == 128 ? 2 : 1;
    constexpr int kStatAt = D == 128 ? 11 : 5, kMoveAt = D == 128 ? 12 : 5;
    auto slot_load = [](int j, int first, int n) { return j >= first && (j - first) % kEvery == 0 && (j - first) / kEvery < n ? (j - first) / kEvery : -1; };
    int stage = 0, it = 0;
    iss_stage = R.startup_tiles;  // also where there are fewer tiles than that
    uint32_t off = 0;
    auto offset = [&](int k) {  // rows past the last query re-read it
      const uint32_t last = min(left_it, kBK) - 1, row = (k >> 1) * 4 * Z::kRowsPerInst;
      if (k & 1) off = min(d_row + row * dstep, last * dstep) + src.y;
      else off = min(q_row + row * D * 2, last * D * 2) + src.y;
    };
    auto load = [&](int k) {
      const uint32_t dst = lds0 + iss_stage * kStageBytes + wave * 1024 + (k >> 1) * 4096;
      if (k & 1) gload_lds16_so(d_it, off, dst + Z::kTileBytes);
      else gload_lds16_so(q_it, off, dst);
    };
    auto stat_offset = [&]() { off = (uint32_t)min(lane, left_it - 1) * 4; };
    auto stat_load = [&]() { gload_lds4_so(s_it, off, ldl0 + (iss_stage * 128 + (wave & 1) * 64) * 4); };
    auto end_tile = [&]() {
      iss_stage = iss_stage == kStages - 1 ? 0 : iss_stage + 1;
      wait_vmcnt<ring::loads_kept_after_iteration(R, true)>();
      // a bare barrier: the reads of this tile have returned (the products above used them), and those of the next tile's
      // first fragments, still on their way, come from a stage that the next iteration does not refill either
      asm volatile("" ::: "memory");
      __builtin_amdgcn_s_barrier();
      asm volatile("" ::: "memory");
    };
    auto run_tiles = [&](auto masked_c, int t_lo, int t_hi) {
      for (int x = (t_hi - t_lo) * rep, t = t_hi - 1, hq = 0; x > 0; --x, ++it) {
        const int nstage = stage == kStages - 1 ? 0 : stage + 1;
        const int i0 = (qt_start + t) * kBK;
        uint32_t tr_next = 0, tra_next[2 * MB];
        bool more = false, wrap = false;
        int64_t q_step = 0, d_step = 0;
        int s_step = 0, left_step = 0;
        step(masked_c, s0, d0, s1, d1, 0, i0,
             [&](int slot) {
               const int j = slot - kA;
               if (slot_load(j, kAt0, kFirst) >= 0) load(slot_load(j, kAt0, kFirst));
               if (j == 0) {
                 more = it + R.issue_ahead + 1 < n_it;  // else the last tile is requested once more
                 wrap = iss_h + 1 == rep;
                 iss_h = !more ? iss_h : wrap ? 0 : iss_h + 1;
               }
               if (j == 1) q_step = more ? (wrap ? q_wrap : q_head) : 0;
               if (j == 2) d_step = more ? (wrap ? d_wrap : d_head) : 0;
               if (j == 3) { s_step = more ? (wrap ? s_wrap : p.Sq) : 0; left_step = more && wrap ? kBK : 0; }
             },
             [&](int slot) {
               const int j = slot - kA;
               if (slot == 0) rm_next = rm_lane + nstage * kStageBytes;
               // k-step ks is read in slot 0, 1, 2 (head_dim 128) or 2 ks - 2
#pragma unroll
               for (int ks = 0; ks < KS; ++ks)
                 if (D == 64 || ks < 2 ? slot == 0 : j == (ks == 2 ? 0 : 2 * ks - 4)) rma[ks] = rm_next ^ (uint32_t)(ks << 5);
               if (j == (D == 128 ? 5 : 3)) st_next = st_lane + nstage * 512;
               if (slot_load(j + 1, kAt0, kFirst) >= 0) offset(slot_load(j + 1, kAt0, kFirst));
             });
        step(masked_c, s1, d1, s0, d0, 1, i0 + 32,
             [&](int slot) {
               const int j = slot - kA, k = slot_load(j, kAt1, kLoads - kFirst);
               if (k >= 0) load(kFirst + k);
               if (j == kStatAt) stat_load();
               if (j == kMoveAt) q_it += q_step;
               if (j == kMoveAt + 1) d_it += d_step;
               if (j == kMoveAt + 2) { s_it += s_step; left_it += left_step; }
             },
             [&](int slot) {
               const int j = slot - kA, k = slot_load(j + 1, kAt1, kLoads - kFirst), x2 = j - (kB / 2 - 2);
               if (j == kB / 2 - 3) tr_next = tr_lane + nstage * kStageBytes;
               if (x2 >= 0 && x2 < 2 * MB) tra_next[x2] = tr_addr(tr_next, x2);
               if (k >= 0) offset(kFirst + k);
               if (j == kStatAt - 1) stat_offset();
             });
        end_tile();
        stage = nstage;
#pragma unroll
        for (int i = 0; i < 2 * MB; ++i) tra[i] = tra_next[i];
        if (++hq == rep) { hq = 0; --t; }
      }
    };
    // Blocks whose queries all lie before this wave's first key are left out (6 of 16 per head in a full workgroup on the diagonal), not
    // computed and masked: 0 times a value that is not finite would reach dV and dK of keys that the query does not see.  The stream ends with
    // them.  Of the tiles [t_none, t_half), one at most, the wave needs the second block (its scores first, then the rest: nothing overlaps),
    // of [0, t_none) nothing: it requests its share and keeps the others company.  What the block before has computed ahead nobody reads.
    // dK/dV, all blocks -> this, us: head_dim 64, 8 x 18 / 6 heads, 2048 tokens 157.1 -> 154.8, 24 x 16 / 4, 1024 121.1 -> 116.5, 96 x 16 / 2, 384 84.0 ->
    // 78.2; head_dim 128 (the others' products of a workgroup that is alone on its CU set the time) 12 x 16 / 4, 2048 373.6 -> 372.7.
    const int before = p.causal ? max(kw0 - p.q_start, 0) : 0;  // queries before the wave's first key
    const int t_none = min(max(before / kBK - qt_start, 0), n_vis), t_half = min(max((before + 32) / kBK - qt_start, 0), n_vis);
    auto request = [&]() {  // a tile's loads outside the slots
#pragma unroll
      for (int k = 0; k < kLoads; ++k) { offset(k); load(k); }
      stat_offset();
      stat_load();
      if (it + R.issue_ahead + 1 < n_it) advance();
    };
    auto run_second_blocks = [&](int t) {
      for (int hq = 0; hq < rep; ++hq, ++it) {  // its fragments and statistics are there, as at the start of every iteration
        const int nstage = stage == kStages - 1 ? 0 : stage + 1;
#pragma unroll
        for (int i = 0; i < kA; ++i) {
          const int o = order(i);
          if (o < KS) mfma32_fixed(s1, qf[o], kreg[o]);
          else mfma32_fixed(d1, df[o - KS], vreg[o - KS]);
        }
        request();
        bf16x8 dT[MB][2], qT[MB][2];
#pragma unroll
        for (int mb = 0; mb < MB; ++mb)
#pragma unroll
          for (int half = 0; half < 2; ++half) {
            dT[mb][half] = frag_tr_at<D>(tra[2 * mb], tra[2 * mb + 1], 2 + half, Z::kTileBytes);
            qT[mb][half] = frag_tr_at<D>(tra[2 * mb], tra[2 * mb + 1], 2 + half, 0);
          }
        mfma32_fixed_done(s1);
        mfma32_fixed_done(d1);
        const int ib = (qt_start + t) * kBK + 32, lo = key - p.q_start - ib - 4 * hh, hi = p.Sq - ib - 4 * hh;
#pragma unroll
        for (int r = 0; r < 16; ++r) {
          const int c = 8 * (r >> 2) + (r & 3);
          if (c < lo || c >= hi) s1[r] = -INFINITY;
          s1[r] = fast_exp2(s1[r]);
          d1[r] *= s1[r];
        }
        bf16x8 pw[2] = {pack_c_half(s1, 0), pack_c_half(s1, 1)}, dw[2] = {pack_c_half(d1, 0), pack_c_half(d1, 1)};
#pragma unroll
        for (int half = 0; half < 2; ++half) { mfma32_settle<false>(pw[half]); mfma32_settle<false>(dw[half]); }
#pragma unroll
        for (int half = 0; half < 2; ++half)
#pragma unroll
          for (int mb = 0; mb < MB; ++mb) {
            mfma32_acc(dvacc[mb], dT[mb][half], pw[half]);
            mfma32_acc(dkacc[mb], qT[mb][half], dw[half]);
          }
        rm_next = rm_lane + nstage * kStageBytes;
        st_next = st_lane + nstage * 512;
#pragma unroll
        for (int ks = 0; ks < KS; ++ks) {
          qf[ks] = swz_frag_rm<D>(rm_next, 1, ks);
          df[ks] = swz_frag_rm<D>(rm_next + Z::kTileBytes, 1, ks);
        }
#pragma unroll
        for (int c = 0; c < 8; ++c) load_stat(s1, d1, st_next, 1, c);
#pragma unroll
        for (int x = 0; x < 2 * MB; ++x) tra[x] = tr_addr(tr_lane + nstage * kStageBytes, x);
        end_tile();
        stage = nstage;
      }
    };
    const int t_inside = min(t_diag, t_full);
    run_tiles(IC<2>{}, t_end, n_vis);
    run_tiles(IC<0>{}, t_diag, t_end);
    run_tiles(IC<2>{}, max(t_half, t_inside), t_diag);
    run_tiles(IC<1>{}, t_half, t_inside);
    if (t_half > t_none) run_second_blocks(t_none);
    asm volatile("s_waitcnt lgkmcnt(0)" ::: "memory");  // fragments requested for a block that is left out: no product waits for them
    for (int x = t_none * rep; x > 0; --x, ++it) {
      request();
      end_tile();
    }
#pragma unroll
    for (int mb = 0; mb < MB; ++mb) { mfma32_acc_done(dvacc[mb]); mfma32_acc_done(dkacc[mb]); }
    static_assert(R.always_requests, "no branch around the loads of an iteration");
    wait_vmcnt<0>();  // the last tile, requested once more, has left the stages that the epilogue uses
    __syncthreads();
  } else {
    auto request_rowmajor = [&](uint32_t rm, int qb) {  // qb is a compile-time constant at every call site
#pragma unroll
      for (int ks = 0; ks < KS; ++ks) {
        qf[ks] = swz_frag_rm<D>(rm, qb, ks);
        df[ks] = swz_frag_rm<D>(rm + Z::kTileBytes, qb, ks);
      }
    };
    // one 32-query block (qb = 0/1, compile-time) of the tile whose stage the pointers address;
    // ib = first query of the block; the row-major fragments of the block after it start at next_rm.
    // The mask variant is compile-time so that a whole block is one straight-line scheduling region:
    // 0 none, 1 causal diagonal only (every query of the block exists), 2 diagonal and / or end of the queries.
    auto step = [&](auto masked_c, uint32_t tr, uint32_t st, int qb, int ib, uint32_t next_rm, int next_qb) {
      constexpr int MASK = decltype(masked_c)::value;
      // head_dim 128 (one wave per SIMD, nothing else to hide the exp2 phase behind): the compiler's interleaving
      // strategy for exp2 work between MFMA chains, measured -3 % on 128-key workgroups; at head_dim 64 it changes nothing
      if constexpr (D == 128) __builtin_amdgcn_iglp_opt(3);
      // accumulators of S and dP start from -lse2 / -delta of the 16 query rows their registers map to
      f32x16 s, dpv;
#pragma unroll
      for (int c = 0; c < 4; ++c) {
        const f32x4 l4 = lds_read_f4(st + (32 * qb + 8 * c) * 4);
        const f32x4 d4 = lds_read_f4(st + (64 + 32 * qb + 8 * c) * 4);
        s[4 * c] = l4[0]; s[4 * c + 1] = l4[1]; s[4 * c + 2] = l4[2]; s[4 * c + 3] = l4[3];
        dpv[4 * c] = d4[0]; dpv[4 * c + 1] = d4[1]; dpv[4 * c + 2] = d4[2]; dpv[4 * c + 3] = d4[3];
      }
#pragma unroll
      for (int ks = 0; ks < KS; ++ks) s = mfma32(qf[ks], kreg[ks], s);
#pragma unroll
      for (int ks = 0; ks < KS; ++ks) dpv = mfma32(df[ks], vreg[ks], dpv);
      bf16x8 dT[MB][2], qT[MB][2];
#pragma unroll
      for (int mb = 0; mb < MB; ++mb) {
        dT[mb][0] = swz_frag_tr<D>(tr + Z::kTileBytes, mb, 2 * qb);
        qT[mb][0] = swz_frag_tr<D>(tr, mb, 2 * qb);
        dT[mb][1] = swz_frag_tr<D>(tr + Z::kTileBytes, mb, 2 * qb + 1);
        qT[mb][1] = swz_frag_tr<D>(tr, mb, 2 * qb + 1);
      }
      if (MASK != 0) {  // block touches the diagonal or the end of the queries
        // register r holds query ib + 4hh + c_r with c_r = 8(r/4) + r%4 a compile-time constant.
        // masked iff key > query + q_start  <=>  c_r < key - q_start - ib - 4hh,   or query >= Sq
        const int t = p.causal ? key - p.q_start - ib - 4 * hh : -1;
        const int u = p.Sq - ib - 4 * hh;
#pragma unroll
        for (int r = 0; r < 16; ++r) {
          const int c = 8 * (r >> 2) + (r & 3);
          if (MASK == 1 ? c < t : (c < t || c >= u)) s[r] = -INFINITY;
        }
      }
#pragma unroll
      for (int r = 0; r < 16; ++r) {
        s[r] = fast_exp2(s[r]);
        dpv[r] *= s[r];
      }
      const bf16x8 p0 = pack_c_half(s, 0), p1 = pack_c_half(s, 1);
      const bf16x8 ds0 = pack_c_half(dpv, 0), ds1 = pack_c_half(dpv, 1);
      request_rowmajor(next_rm, next_qb);  // unconditional: past the last block the fragments are simply unused
#pragma unroll
      for (int mb = 0; mb < MB; ++mb) {
        dvacc[mb] = mfma32(dT[mb][0], p0, dvacc[mb]);
        dkacc[mb] = mfma32(qT[mb][0], ds0, dkacc[mb]);
      }
#pragma unroll
      for (int mb = 0; mb < MB; ++mb) {
        dvacc[mb] = mfma32(dT[mb][1], p1, dvacc[mb]);
        dkacc[mb] = mfma32(qT[mb][1], ds1, dkacc[mb]);
      }
    };

    // ---- pipeline start-up: tiles 0 and 1 have landed (first wait above), tile 2 is in flight
    if (n_it > 0) request_rowmajor(rm_lane, 0);
    int stage = 0, it = 0;
    auto run_tiles = [&](auto masked_c, int t_lo, int t_hi) {
      constexpr int MASK = decltype(masked_c)::value;
      for (int t = t_lo; t < t_hi; ++t, ++it) {
        const int nstage = stage == kStages - 1 ? 0 : stage + 1;
        const int i0 = (qt_start + t) * kBK;
        const uint32_t rm = rm_lane + stage * kStageBytes, tr = tr_lane + stage * kStageBytes;
        const uint32_t st = st_lane + stage * 512;
        // on the diagonal a block whose last query still lies before this wave's first key is masked entirely:
        // it only passes the fragment request on (wave-uniform, so the barrier below is reached all the same)
        if constexpr (PARTS == 1) {
          if (MASK == 1 && kw0 > i0 + 31 + p.q_start) request_rowmajor(rm, 1); else step(masked_c, tr, st, 0, i0, rm, 1);
          if (MASK == 1 && kw0 > i0 + 63 + p.q_start) request_rowmajor(rm_lane + nstage * kStageBytes, 0);
          else step(masked_c, tr, st, 1, i0 + 32, rm_lane + nstage * kStageBytes, 0);
        } else {
          const int ib = i0 + 32 * part;
          if (MASK == 1 && kw0 > ib + 31 + p.q_start) request_rowmajor(rm_lane + nstage * kStageBytes, 0);
          else step(masked_c, tr, st, 0, ib, rm_lane + nstage * kStageBytes, 0);
        }
        if (it + R.issue_ahead < n_it) { issue_next(); wait_vmcnt<ring::loads_kept_after_iteration(R, true)>(); } else wait_vmcnt<ring::loads_kept_after_iteration(R, false)>();
        __syncthreads();
        stage = nstage;
      }
    };
    for (int hq = 0; hq < rep; ++hq) {
      run_tiles(IC<1>{}, 0, min(t_diag, t_full));
      run_tiles(IC<2>{}, min(t_diag, t_full), t_diag);
      run_tiles(IC<0>{}, t_diag, t_end);
      run_tiles(IC<2>{}, t_end, n_vis);
    }
  }

  // ---- epilogue: lane = key row, registers = head-dim entries.  The rows it reads (the raw key for the normaliser's
  // gradient, with a value residual the raw v and v_first rows for the coefficient gradients) come in like the
  // prologue's rows: as 128-row blocks by direct loads into the ring's stages, which are idle now (every wave has
  // passed the last iteration's barrier), and from there in the accumulators' layout.  Read row-per-lane from global
  // memory, 8 bytes per lane, every wave-wide load would touch 32 cache lines and the three tensors would keep the
  // address path of the vector memory unit busy for 4-12 us of the launch.
  static_assert(R.epilogue_row_stages == (PARTS == 1 ? 3 : 2), "k, v, v_first blocks in stages 0, 1, 2; or in three tiles of stages 0 and 1");
  const bool live = key < p.Sk;
  float c1 = 1.f, c2 = 0.f;
  if (p.vr_coef) { c1 = p.vr_coef[0]; c2 = p.vr_coef[1]; }
  u32x2 kraw[MB][4], vraw[MB][4], fraw[MB][4];
  {
    const int rows_left = min(p.Sk - k0, BKV);
    const uint32_t wave_dst = lds0 + wave * 1024;
    const char* kb = reinterpret_cast<const char*>(row_ptr<uint16_t>(p.k, b, g, k0));
    const char* vb = p.vr_coef ? reinterpret_cast<const char*>(row_ptr<uint16_t>(p.v, b, g, k0)) : kb;
    const char* fb = p.vr_coef ? reinterpret_cast<const char*>(row_ptr<uint16_t>(p.v_first, b, g, k0)) : kb;
    const uint32_t kst = (uint32_t)p.k.stride_s * 2, vst = p.vr_coef ? (uint32_t)p.v.stride_s * 2 : kst, fst = (uint32_t)p.v_first.stride_s * 2;
    if constexpr (PARTS == 1) {
      issue_tile_pair<D>(kb, kb, rowblock_lane_offsets<D>(kst, 0, rows_left, src.x, src.y), wave_dst);
      if (p.vr_coef) {
        issue_tile_pair<D>(vb, vb, rowblock_lane_offsets<D>(vst, 0, rows_left, src.x, src.y), wave_dst + kStageBytes);
        issue_tile_pair<D>(fb, fb, rowblock_lane_offsets<D>(fst, 0, rows_left, src.x, src.y), wave_dst + 2 * kStageBytes);
      }
    } else {  // 64 rows each: the two tiles of stage 0 and the first of stage 1
      issue_tile_pair<D>(kb, vb, tile_lane_offsets<D>(kst, vst, rows_left, src.x, src.y), wave_dst);
      if (p.vr_coef) issue_tile_pair<D>(fb, fb, tile_lane_offsets<D>(fst, fst, rows_left, src.x, src.y), wave_dst + kStageBytes);
      // The two parts of a key block meet here: part 0 finishes dK, part 1 dV, so each hands the other's half over
      // through the idle stages 2 and 3 (one slot per wave, 16 bytes per lane and access: conflict-free).
      static_assert(4 * MB * 4096 <= R.merge_stages * kStageBytes, "one accumulator per wave in two stages");
      char* const slot = lds + R.merge_stage_first * kStageBytes + lane * 16;
#pragma unroll
      for (int mb = 0; mb < MB; ++mb)
#pragma unroll
        for (int c = 0; c < 4; ++c) {
          f32x4 t;
#pragma unroll
          for (int i = 0; i < 4; ++i) t[i] = part == 0 ? dvacc[mb][4 * c + i] : dkacc[mb][4 * c + i];
          *reinterpret_cast<f32x4*>(slot + wave * (MB * 4096) + (4 * mb + c) * 1024) = t;
        }
    }
    wait_vmcnt<0>();
    __syncthreads();
    if constexpr (PARTS == 2) {
      const char* const other = lds + R.merge_stage_first * kStageBytes + lane * 16 + (wave ^ kKeyWaves) * (MB * 4096);
#pragma unroll
      for (int mb = 0; mb < MB; ++mb)
#pragma unroll
        for (int c = 0; c < 4; ++c) {
          const f32x4 t = *reinterpret_cast<const f32x4*>(other + (4 * mb + c) * 1024);
#pragma unroll
          for (int i = 0; i < 4; ++i) { dvacc[mb][4 * c + i] += t[i]; dkacc[mb][4 * c + i] += t[i]; }  // each uses its own one only
        }
    }
    // rows 32*key_wave .. +31 of a block: half (key_wave >> 1) of its stage, row block (key_wave & 1) of that tile
    constexpr int kVRows = PARTS == 1 ? kStageBytes : Z::kTileBytes, kFRows = PARTS == 1 ? 2 * kStageBytes : kStageBytes;
    const uint32_t ct = lds0 + (key_wave >> 1) * Z::kTileBytes + swz_off_ct<D>(lane) + (key_wave & 1) * 32 * Z::kRB;
#pragma unroll
    for (int mb = 0; mb < MB; ++mb)
#pragma unroll
      for (int c = 0; c < 4; ++c) {
        const uint32_t off = (uint32_t)((4 * mb + c) << 4);
        kraw[mb][c] = lds_read8(ct ^ off);
        if (p.vr_coef) {
          vraw[mb][c] = lds_read8((ct + kVRows) ^ off);
          fraw[mb][c] = lds_read8((ct + kFRows) ^ off);
        }
      }
  }
  RopeCt<MB> rope_ct;
  if (ROPE) {
    const int64_t pos = (int64_t)(p.rope_k_pos0 + key_c) * (D / 2);
    rope_ct = rope_ct_load<MB>(p.rope_cos + pos, p.rope_sin + pos, hh);
  }
  const bool own_dk = PARTS == 1 || part == 0, own_dv = PARTS == 1 || part == 1;
  if (own_dv) {
    uint16_t* ovp = row_ptr_mut<uint16_t>(p.dv, b, g, key_c);
#pragma unroll
    for (int mb = 0; mb < MB; ++mb) {
      float val[16];
#pragma unroll
      for (int r = 0; r < 16; ++r) val[r] = c1 * dvacc[mb][r];
      store_ct_block(ovp, mb, hh, live, val);
    }
  }
  if (p.vr_coef) {
    float s1 = 0.f, s2 = 0.f;
    if (own_dv) {
      uint16_t* ofp = row_ptr_mut<uint16_t>(p.dv_first, b, g, key_c);
#pragma unroll
      for (int mb = 0; mb < MB; ++mb) {
        float val[16], vv[16], ff[16];
#pragma unroll
        for (int r = 0; r < 16; ++r) val[r] = c2 * dvacc[mb][r];
        store_ct_block(ofp, mb, hh, live, val);
        unpack_ct_block(vraw[mb], vv);
        unpack_ct_block(fraw[mb], ff);
#pragma unroll
        for (int r = 0; r < 16; ++r)
          if (live) { s1 += dvacc[mb][r] * vv[r]; s2 += dvacc[mb][r] * ff[r]; }
      }
    }
#pragma unroll
    for (int o = 1; o < 64; o <<= 1) { s1 += __shfl_xor(s1, o, 64); s2 += __shfl_xor(s2, o, 64); }
    if (lane == 0) { red[wave * 2] = s1; red[wave * 2 + 1] = s2; }
    __syncthreads();
    if (tid < 2) a.dcoef_part[(int64_t)bid * 2 + tid] = red[tid] + red[2 + tid] + red[4 + tid] + red[6 + tid];
  }
  // dk through the normaliser: W = ln2 * dkacc = dL/dKhat (natural units), dk = b W - (b^3/D)(W.k) k
  if (own_dk) {
    float kv[MB][16];
#pragma unroll
    for (int mb = 0; mb < MB; ++mb) unpack_ct_block(kraw[mb], kv[mb]);
    // the normaliser acted on the rotated key: work in that frame, rotate the gradient back
    if (ROPE) rope_ct_apply<MB, false>(kv, rope_ct);
    float dot = 0.f, ss = 0.f;
#pragma unroll
    for (int mb = 0; mb < MB; ++mb)
#pragma unroll
      for (int r = 0; r < 16; ++r) { dot += dkacc[mb][r] * kv[mb][r]; ss += kv[mb][r] * kv[mb][r]; }
    dot = half_sum(dot) * kLn2;
    ss = half_sum(ss);
    const float beta = row_normaliser_fast(p, ss, 1.0f / D);
    const float b3 = norm_grad_coef(p, beta, 1.0f / D) * dot;
    uint16_t* okp = row_ptr_mut<uint16_t>(p.dk, b, g, key_c);
    float val[MB][16];
#pragma unroll
    for (int mb = 0; mb < MB; ++mb)
#pragma unroll
      for (int r = 0; r < 16; ++r) val[mb][r] = beta * kLn2 * dkacc[mb][r] - b3 * kv[mb][r];
    if (ROPE) rope_ct_apply<MB, true>(val, rope_ct);
#pragma unroll
    for (int mb = 0; mb < MB; ++mb) store_ct_block(okp, mb, hh, live, val[mb]);
  }
}

template <int D, bool ROPE>
void launch_dkdv_t(const KArgs& a, hipStream_t st) {
  const dim3 grid((unsigned)(bf16_dkdv_grid(a.p) + 1));
  if (dkdv_pipelined(a.p)) hipLaunchKernelGGL((bwd_dkdv_bf16_kernel<D, ROPE, 1, true>), grid, dim3(kThreadsM), 0, st, a);
  else if (dkdv_parts(a.p) == 2) hipLaunchKernelGGL((bwd_dkdv_bf16_kernel<D, ROPE, 2, false>), grid, dim3(kThreadsM), 0, st, a);
  else if constexpr (D == 64) hipLaunchKernelGGL((bwd_dkdv_bf16_kernel<D, ROPE, 1, false>), grid, dim3(kThreadsM), 0, st, a);
}

template <int D, bool ROPE>
void launch_dq_t(const KArgs& a, hipStream_t st) {
  const dim3 grid((unsigned)bf16_dq_grid(a.p));
  if (dq_pipelined(a.p)) hipLaunchKernelGGL((bwd_dq_bf16_kernel<D, ROPE, 1, true>), grid, dim3(kThreadsM), 0, st, a);
  else if (dq_parts(a.p) == 2) hipLaunchKernelGGL((bwd_dq_bf16_kernel<D, ROPE, 2, false>), grid, dim3(kThreadsM), 0, st, a);
  else if constexpr (D == 64) hipLaunchKernelGGL((bwd_dq_bf16_kernel<D, ROPE, 1, false>), grid, dim3(kThreadsM), 0, st, a);
}

}  // namespace

// workgroups of the two launches (the dK/dV launch has one more, its extra reducing workgroup): the workspace holds one
// row of partial sums per workgroup, idle padding workgroups included
int bf16_dq_grid(const segpt_attn_params& p) {
  const int rows = kBwdRows / dq_parts(p);
  return wg_grid((p.Sq + rows - 1) / rows, p.B, p.Hkv, p.H / p.Hkv, wg_pinned_pairs(p.B, p.Hkv, false));
}
int bf16_dkdv_grid(const segpt_attn_params& p) {
  const int rows = kBwdRows / dkdv_parts(p);
  return wg_grid((p.Sk + rows - 1) / rows, p.B, p.Hkv, 1, dkdv_pinned(p));
}

int launch_bwd_dkdv_bf16(const KArgs& a, hipStream_t st) {
  const bool rope = a.p.rope_cos != nullptr;
  if (a.p.D == 64) rope ? launch_dkdv_t<64, true>(a, st) : launch_dkdv_t<64, false>(a, st);
  else if (a.p.D == 128) rope ? launch_dkdv_t<128, true>(a, st) : launch_dkdv_t<128, false>(a, st);
  else return (int)hipErrorInvalidValue;
  return (int)hipGetLastError();
}

int launch_bwd_dq_bf16(const KArgs& a, hipStream_t st) {
  const bool rope = a.p.rope_cos != nullptr;
  if (a.p.D == 64) rope ? launch_dq_t<64, true>(a, st) : launch_dq_t<64, false>(a, st);
  else if (a.p.D == 128) rope ? launch_dq_t<128, true>(a, st) : launch_dq_t<128, false>(a, st);
  else return (int)hipErrorInvalidValue;
  return (int)hipGetLastError();
}

}  // namespace segpt
