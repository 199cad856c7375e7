// fp32 forward and backward on the bf16 matrix pipe: every fp32 operand as the sum of three bf16 numbers.
//
// x = x0 + x1 + x2 with x0 = bf16(x), x1 = bf16(x - x0), x2 = bf16(x - x0 - x1) (round to nearest: 24 bits and the signs of
// the remainders, so the sum is x itself).  The method is Henry, Tang and Heinecke's, "Leveraging the bfloat16 Artificial Intelligence
// Datatype for Higher-Precision Computations" (2019).  A product of two such numbers is six matrix instructions, x0 y0 + (x0 y1 + x1 y0 +
// x1 y1 + x0 y2 + x2 y0), each product exact and summed in fp32; what is left out is below 2^-24 of |x y|.  v_mfma_f32_32x32x16_bf16 does eight times the products of
// v_mfma_f32_32x32x2_f32 in half the time, so six of them take 3/8 of the fp32 instructions' time, and a sum of 64 products is 4 (and
// 20 small ones) roundings deep instead of 32: norm-wise distance of a 32x32 tile of products to float64, 64 / 128 columns:
// fp32 instructions 1.5e-7 / 1.95e-7, one accumulator for all six 1.1e-7 / 1.6e-7, the largest product on its own 4.9e-8 / 6.4e-8.
//
// Range: the last bits of a value below 2^-109 are none of bf16's any more.  Operand tiles with such values are kept with scaled parts
// and take a slower form of the products (see kPart).  Infinities and finite values beyond bf16's largest: see split8.
//
// What that takes: nothing may be split inside a loop that runs once per pair of tiles.  A pre-pass rotates, normalises
// and splits every row once and leaves 32-row tiles as matrix-instruction operands, 1 KB (64 lanes x 16 bytes) each, in the order they
// are used: [unit][x0, x1, x2], D / 16 units a tile.
//   rm  (contraction over the columns): unit u, lane (ln, hh): columns 16 u + 8 hh .. + 7 of row ln.
//   tr  (contraction over the rows): unit 2 mb + s: column MB ln + mb (MB = D / 32) of the rows 16 s + 8 (i / 4) + 4 hh + i % 4,
//       i = 0..7, which are the rows that registers 8 s .. 8 s + 7 of a C tile hold: scores need no shuffle to be the other operand.
// The streamed operands then travel from the L2 straight into registers, without LDS, without a barrier in the loops; the 32
// stationary rows of a workgroup lie in LDS once for its four waves, which share out the streamed tiles as in f32_path.hip.
//
// What bounds it: the streamed tiles, 24 / 36 / 48 KB (forward / dQ / dK/dV at head_dim 64) per 32x32 scores and wave, of which a
// CU gets about 19 bytes a cycle (11 TB/s) whether they are hits in the L2 or requests of a deeper look-ahead: matrix pipe 27 % busy,
// and neither forming the next scores beside this tile's exponentials nor two accumulators more for shorter chains of dependent
// products moved a kernel.  Kernels, us, fp32 instructions -> here: 2 x 8 / 4 heads, 1000 tokens of 64 forward 37 -> 6.9 + 23, dQ and dK/dV 47 +
// 62 -> 60, the pre-pass of the backward 13; the step 143 -> 99.  8 x 18 / 6 heads of 2048 tokens 3453 -> 2250, 1 x 4 / 2 heads of 1000 x
// 128 213 -> 117.
#include <algorithm>

#include "f32_common.hpp"

namespace segpt {
namespace {

typedef __bf16 bf16x8 __attribute__((ext_vector_type(8)));
typedef uint32_t u32x4 __attribute__((ext_vector_type(4)));

constexpr int kUnitBytes = 3 * 1024;
template <int D>
constexpr int kUnits = D / 16;
template <int D>
constexpr int kTileBytes = kUnits<D> * kUnitBytes;

struct Split3 {
  bf16x8 p[3];
};
// The streamed tiles come in as halves of 32 columns (rm) or of one block mb (tr), two units each, MB = D / 32 halves a
// tile: twelve matrix instructions (384 cycles).
struct Half {
  Split3 u[2];
};
constexpr int kHalfBytes = 2 * kUnitBytes;

// where the pre-pass leaves its tiles
struct SplitMap {
  char *k_rm, *v, *k_tr, *q_rm, *q_tr, *d_rm, *d_tr;  // v: tr for the forward, rm for the backward
  float* stat;                                        // [B * H][query tiles][lse of 32 rows, delta of 32 rows]
  uint32_t *k_small, *v_small, *q_small, *d_small;    // a tile's parts are scaled (kPart)
};
__device__ __forceinline__ int tiles_of(int n) { return (n + kRows - 1) / kRows; }
template <int D>
__device__ __forceinline__ SplitMap split_map(const KArgs& a, bool bwd) {
  const int64_t kvt = (int64_t)a.p.B * a.p.Hkv * tiles_of(a.p.Sk), qt = bwd ? (int64_t)a.p.B * a.p.H * tiles_of(a.p.Sq) : 0;
  const int64_t kv = kvt * kTileBytes<D>, q = qt * kTileBytes<D>;
  SplitMap m;
  m.k_rm = a.f32_split;
  m.v = m.k_rm + kv;
  m.k_tr = m.v + kv;  // from here on to stat: backward only
  m.q_rm = m.k_tr + (bwd ? kv : 0);
  m.q_tr = m.q_rm + q;
  m.d_rm = m.q_tr + q;
  m.d_tr = m.d_rm + q;
  m.stat = reinterpret_cast<float*>(m.d_tr + q);
  m.k_small = reinterpret_cast<uint32_t*>(m.stat + qt * 64);
  m.v_small = m.k_small + kvt;
  m.q_small = m.v_small + kvt;
  m.d_small = m.q_small + qt;
  return m;
}

// Nothing is scheduled across: every half is requested two steps before its use and not earlier.  Left to itself the compiler
// hoists a whole iteration's requests and spills (dQ and dK/dV at head_dim 64: 72 and 112 registers).
__device__ __forceinline__ void step_end() { __builtin_amdgcn_sched_barrier(0); }

__device__ __forceinline__ f32x16 mfma16(bf16x8 a, bf16x8 b, f32x16 c) { return __builtin_amdgcn_mfma_f32_32x32x16_bf16(a, b, c, 0, 0, 0); }

// Beyond bf16's range: a finite value there keeps bf16's largest number as its first part, the rest goes into the other two.  An infinity is
// the third part alone, which meets only the other operand's first part: the product is that infinity, or NaN where the other
// operand is 0, as with the fp32 instructions (as the first part it met the remainders of either sign).
constexpr float kBf16Max = 3.38953139e38f;
template <int N>
__device__ __forceinline__ bool beyond_bf16(const float (&x)[N]) {
  float m = 0.f;
#pragma unroll
  for (int i = 0; i < N; ++i) m = fmaxf(m, fabsf(x[i]));  // NaN needs nothing: every part of it is NaN
  return __builtin_amdgcn_ballot_w64(m > kBf16Max) != 0;
}
// Small values: the second part of a value is up to 2^16, the third up to 2^24 below it.  Where bits would fall below bf16's last, 2^-133, the
// second part is kept times kPart and the third times kPart^2, and no bit is lost whose product fp32 could hold.  That is a property of
// a tile (its flag in SplitMap); a wave that meets such a tile takes all its tiles through a loop of its own, in which the products of each
// scale are formed apart.  dO of 1e-35: gradients were 6e-5 from float64, now 3.4e-7 (fp32 instructions 4e-7).  The flags and split_lanes
// cost 1 to 4 % (backward of 2 x 8 / 4 heads, 1000 tokens 75.9 -> 78.1 us); scaling always and no second loop cost 5 to 8 %.  The same call with
// one such row: 97, with v and dO of 1e-33: 106, its forward 28 -> 49 (fp32 instructions 111 and 36).
constexpr float kPart = 128.f, kSmall = 7.888609052e-31f;  // 2^-100
__device__ __forceinline__ bool any_lane(bool x) { return __builtin_amdgcn_ballot_w64(x) != 0; }
__device__ __forceinline__ bool is_small(float x) { return x != 0.f && fabsf(x) < kSmall; }
template <bool BEYOND>
__device__ __forceinline__ Split3 split8(const float (&x)[8], float part) {
  Split3 s;
  u32x4 w[3];
#pragma unroll
  for (int i = 0; i < 4; ++i) {
    float v[2] = {x[2 * i], x[2 * i + 1]}, first[2] = {v[0], v[1]};
    if (BEYOND) {
#pragma unroll
      for (int e = 0; e < 2; ++e) {
        const bool inf = __builtin_isinf(v[e]);
        first[e] = inf ? 0.f : fabsf(v[e]) > kBf16Max ? copysignf(kBf16Max, v[e]) : v[e];
      }
    }
    w[0][i] = pack_bf16x2(first[0], first[1]);
    const float a = (v[0] - bf16lo(w[0][i])) * part, b = (v[1] - bf16hi(w[0][i])) * part;
    if (BEYOND) {
      w[1][i] = pack_bf16x2(__builtin_isinf(v[0]) ? 0.f : a, __builtin_isinf(v[1]) ? 0.f : b);
    } else {
      w[1][i] = pack_bf16x2(a, b);
    }
    w[2][i] = pack_bf16x2((a - bf16lo(w[1][i])) * part, (b - bf16hi(w[1][i])) * part);
  }
#pragma unroll
  for (int k = 0; k < 3; ++k) s.p[k] = __builtin_bit_cast(bf16x8, w[k]);
  return s;
}
__device__ __forceinline__ Split3 split_row(const float (&x)[8], float part) { return beyond_bf16(x) ? split8<true>(x, part) : split8<false>(x, part); }

__device__ __forceinline__ Split3 load_unit(const char* unit, int lane) {
  Split3 s;
#pragma unroll
  for (int k = 0; k < 3; ++k) s.p[k] = *reinterpret_cast<const bf16x8*>(unit + k * 1024 + lane * 16);
  return s;
}
__device__ __forceinline__ Half load_half(const char* half, int lane) { return {{load_unit(half, lane), load_unit(half + kUnitBytes, lane)}}; }
__device__ __forceinline__ void store_unit(char* unit, const Split3& s, int lane) {
#pragma unroll
  for (int k = 0; k < 3; ++k) *reinterpret_cast<bf16x8*>(unit + k * 1024 + lane * 16) = s.p[k];
}

// any small value in the tile that a wave holds?
template <int D>
__device__ __forceinline__ bool tile_small(const f32x4v (&x)[T32<D>::kPasses]) {
  uint32_t m = ~0u;
#pragma unroll
  for (int ps = 0; ps < T32<D>::kPasses; ++ps)
#pragma unroll
    for (int e = 0; e < 4; ++e) m = min(m, (__float_as_uint(x[ps][e]) << 1) - 1);  // the sign goes, zero becomes the largest
  return any_lane(m < (__float_as_uint(kSmall) << 1) - 1);
}
// the flags of n tiles; the first 64 are requested early
__device__ __forceinline__ uint32_t first_flags(const uint32_t* flags, int n, int lane) { return lane < n ? flags[lane] : 0; }
__device__ __forceinline__ bool any_small(uint32_t first, const uint32_t* flags, int n, int lane) {
  for (int i = lane + 64; i < n; i += 64) first |= flags[i];
  return any_lane(first);
}
// units u0, u0 + step, ... of a row-major fp32 tile in LDS
template <int D>
__device__ __forceinline__ void emit_rm(const float* tile, char* dst, int lane, float part, int u0 = 0, int step = 1) {
  for (int u = u0; u < kUnits<D>; u += step) {
    const f32x4v* src = reinterpret_cast<const f32x4v*>(tile + (lane & 31) * T32<D>::kRS + 16 * u + 8 * (lane >> 5));
    const f32x4v lo = src[0], hi = src[1];
    const float x[8] = {lo[0], lo[1], lo[2], lo[3], hi[0], hi[1], hi[2], hi[3]};
    store_unit(dst + u * kUnitBytes, split_row(x, part), lane);
  }
}
template <int D>
__device__ __forceinline__ void emit_tr(const float* tile, char* dst, int lane, float part) {
  constexpr int MB = T32<D>::kMB;
#pragma unroll
  for (int u = 0; u < kUnits<D>; ++u) {
    const float* src = tile + MB * (lane & 31) + u / 2;
    float x[8];
#pragma unroll
    for (int i = 0; i < 8; ++i) x[i] = src[crow(8 * (u % 2) + i, lane >> 5) * T32<D>::kRS];
    store_unit(dst + u * kUnitBytes, split_row(x, part), lane);
  }
}

// the five small products of a pair and the large one, into accumulators of their own or into one
__device__ __forceinline__ f32x16 small5(const Split3& a, const Split3& b, f32x16 c) {
  c = mfma16(a.p[0], b.p[2], c);
  c = mfma16(a.p[2], b.p[0], c);
  c = mfma16(a.p[1], b.p[1], c);
  c = mfma16(a.p[0], b.p[1], c);
  return mfma16(a.p[1], b.p[0], c);
}
// the same where the second parts of a, b or both are scaled by 1 / fa, 1 / fb, the third parts by the squares
__device__ __forceinline__ f32x16 scaled5(const Split3& a, float fa, const Split3& b, float fb, f32x16 c) {
  const int ia[5] = {0, 2, 1, 0, 1}, ib[5] = {2, 0, 1, 1, 0};
  const float f[5] = {fb * fb, fa * fa, fa * fb, fb, fa};
#pragma unroll
  for (int i = 0; i < 5; ++i) {
    const f32x16 t = mfma16(a.p[ia[i]], b.p[ib[i]], zero16());
#pragma unroll
    for (int r = 0; r < 16; ++r) c[r] = fmaf(t[r], f[i], c[r]);
    step_end();  // one product's 16 registers at a time
  }
  return c;
}
// what a tile's *_small flag means for its products (wave-uniform)
__device__ __forceinline__ float part_scale(bool small) { return small ? 1.f / kPart : 1.f; }
// X . B^T over the columns: C rows = rows of the streamed tile, C columns = the 32 stationary rows, whose rm units lie in LDS
struct Dot {
  f32x16 large = zero16(), small = zero16();
  __device__ __forceinline__ void add(const Half& a, const char* b_lds, int lane) {
#pragma unroll
    for (int u = 0; u < 2; ++u) {
      const Split3 b = load_unit(b_lds + u * kUnitBytes, lane);
      small = small5(a.u[u], b, small);
      large = mfma16(a.u[u].p[0], b.p[0], large);
    }
  }
  // the same for all units of a streamed tile, which come in one by one
  template <int D>
  __device__ __forceinline__ void add_scaled(const char* a_tile, bool a_small, const char* b_lds, bool b_small, int lane) {
    const float fa = part_scale(a_small), fb = part_scale(b_small);
#pragma unroll 1
    for (int u = 0; u < kUnits<D>; ++u) {
      const Split3 a = load_unit(a_tile + u * kUnitBytes, lane), b = load_unit(b_lds + u * kUnitBytes, lane);
      small = scaled5(a, fa, b, fb, small);
      large = mfma16(a.p[0], b.p[0], large);
    }
  }
  __device__ __forceinline__ f32x16 sum() const {
    f32x16 s;
#pragma unroll
    for (int r = 0; r < 16; ++r) s[r] = large[r] + small[r];
    return s;
  }
};
// scores (registers = rows of the streamed tile) as the other operand of the product over those rows
struct Scores3 {
  Split3 s[2];
};
template <bool BEYOND>
__device__ __forceinline__ Scores3 split16(const f32x16& w, float part) {
  Scores3 b;
#pragma unroll
  for (int s = 0; s < 2; ++s) {
    const float x[8] = {w[8 * s], w[8 * s + 1], w[8 * s + 2], w[8 * s + 3], w[8 * s + 4], w[8 * s + 5], w[8 * s + 6], w[8 * s + 7]};
    b.s[s] = split8<BEYOND>(x, part);
  }
  return b;
}
// Probabilities or, GRADS, their gradients.  The scores of a column (a lane and the one 32 on) add up among themselves: where the largest of
// them is small, all are taken 2^64 times as large and their sum is multiplied by f.  (The forward's need no look, a row's largest is or was 1.)
struct LaneScores {
  Scores3 s;
  float f;
};
template <bool GRADS>
__device__ __forceinline__ LaneScores split_lanes(f32x16& w) {
  float m = 0.f;
#pragma unroll
  for (int r = 0; r < 16; ++r) m = fmaxf(m, fabsf(w[r]));  // NaN needs nothing: every part of it is NaN
  m = half_max(m);  // two lanes hold a column
  LaneScores x;
  x.f = 1.f;
  f32x16 v = w;
  if (any_lane(is_small(m))) {
    const bool up = is_small(m);
    x.f = up ? 0x1p-64f : 1.f;
    const float f = up ? 0x1p64f : 1.f;
#pragma unroll
    for (int r = 0; r < 16; ++r) v[r] *= f;
  }
  x.s = GRADS && any_lane(m > kBf16Max) ? split16<true>(v, 1.f) : split16<false>(v, 1.f);
  return x;
}
// acc += (block mb of a tile)^T . w over the 32 rows; the tile's sum is formed by itself and added once
__device__ __forceinline__ f32x16 add_large(const Half& a, const Scores3& w, f32x16 t) {
  t = mfma16(a.u[0].p[0], w.s[0].p[0], t);
  return mfma16(a.u[1].p[0], w.s[1].p[0], t);
}
__device__ __forceinline__ void add_tr(const Half& a, const Scores3& w, f32x16& acc, float f = 1.f) {
  const f32x16 t = add_large(a, w, small5(a.u[1], w.s[1], small5(a.u[0], w.s[0], zero16())));
#pragma unroll
  for (int r = 0; r < 16; ++r) acc[r] = fmaf(t[r], f, acc[r]);
}
__device__ __forceinline__ void add_tr_scaled(const Half& a, bool a_small, const Scores3& w, f32x16& acc) {  // w: always scaled
  const float fa = part_scale(a_small), fw = 1.f / kPart;
  const f32x16 t = add_large(a, w, scaled5(a.u[1], fa, w.s[1], fw, scaled5(a.u[0], fa, w.s[0], fw, zero16())));
#pragma unroll
  for (int r = 0; r < 16; ++r) acc[r] += t[r];
}

// ---- pre-pass: one wave per (tile, tensor, layout).  Forward: keys rm, values tr.  Backward: query and dO tiles in both layouts
// first (four waves of a workgroup on one query tile), then keys rm, keys tr, values rm; the wave of dO's rm tile also owns
// what belongs to a query row: delta = rowsum(dY o Y), dgate, and the gate factor goes into dO here.
template <int D, bool BWD>
__global__ __launch_bounds__(kThreads) void split_prep_kernel(KArgs a) {
  const segpt_attn_params& p = a.p;
  using T = T32<D>;
  __shared__ __attribute__((aligned(16))) float tiles[kWaves][T::kTile];
  const int lane = threadIdx.x & 63;
  const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
  const SplitMap m = split_map<D>(a, BWD);
  const int n_qt = tiles_of(p.Sq), n_kt = tiles_of(p.Sk);
  float* tile = tiles[wave];
  int64_t job = (int64_t)blockIdx.x * kWaves + wave;
  const int64_t q_jobs = BWD ? (int64_t)p.B * p.H * n_qt * 4 : 0;
  f32x4v x[T::kPasses];
  if (BWD && job < q_jobs) {
    const int kind = (int)(job & 3);
    const int64_t t = job >> 2;
    const int qt = (int)(t % n_qt), hb = (int)(t / n_qt), b = hb / p.H, h = hb % p.H, q0 = qt * kRows;
    if (kind < 2) {
      load_tile<D>(x, row_ptr<float>(p.q, b, h, 0), p.q.stride_s, q0, p.Sq, lane);
      f32x4v gs;
#pragma unroll
      for (int e = 0; e < 4; ++e) gs[e] = gprod<D>(p, 4 * (lane % T::kLPR) + e) * p.sm_scale * kLog2e;
      stage_norm<D, true, true>(p, x, gs, p.rope_q_pos0 + q0, p.Sq - 1 - q0, tile, lane);
    } else {
      load_tile<D>(x, row_ptr<float>(p.d_o, b, h, 0), p.d_o.stride_s, q0, p.Sq, lane);
      f32x4v y[T::kPasses];
      if (kind == 2) load_tile<D>(y, row_ptr<float>(p.o, b, h, 0), p.o.stride_s, q0, p.Sq, lane);
#pragma unroll
      for (int ps = 0; ps < T::kPasses; ++ps) {
        const int row = ps * T::kRPP + lane / T::kLPR;
        float sg = 0.f;
        if (p.gate.ptr) sg = sigmoidf_acc(gate_logit(p, b, h, min(q0 + row, p.Sq - 1)));
        if (kind == 2) {
          const f32x4v d = x[ps] * y[ps];
          const float delta = row_sum<T::kLPR>((d[0] + d[1]) + (d[2] + d[3]));
          if (lane % T::kLPR == 0) {
            m.stat[t * 64 + row] = p.lse[((int64_t)b * p.H + h) * p.Sq + min(q0 + row, p.Sq - 1)];
            m.stat[t * 64 + 32 + row] = delta;
            if (p.gate.ptr && q0 + row < p.Sq)
              reinterpret_cast<float*>(p.dgate.ptr)[(int64_t)b * p.dgate.stride_b + (int64_t)(q0 + row) * p.dgate.stride_s + (int64_t)h * p.dgate.stride_h] = (1.0f - sg) * delta;
          }
        }
        if (p.gate.ptr) x[ps] *= p.gate_scale * sg;
      }
      stage_plain<D>(x, tile, lane);
    }
    wave_sync();
    char* const dst = (kind == 0 ? m.q_rm : kind == 1 ? m.q_tr : kind == 2 ? m.d_rm : m.d_tr) + t * kTileBytes<D>;
    const bool small = tile_small<D>(x);
    if (!(kind & 1) && lane == 0) (kind ? m.d_small : m.q_small)[t] = small;
    if (kind & 1) emit_tr<D>(tile, dst, lane, small ? kPart : 1.f);
    else emit_rm<D>(tile, dst, lane, small ? kPart : 1.f);
    return;
  }
  job -= q_jobs;
  constexpr int kKinds = BWD ? 3 : 2;
  const int kind = (int)(job % kKinds);
  const int64_t t = job / kKinds;
  if (t >= (int64_t)p.B * p.Hkv * n_kt) return;
  const int kt = (int)(t % n_kt), bg = (int)(t / n_kt), b = bg / p.Hkv, g = bg % p.Hkv, j0 = kt * kRows;
  const bool values = kind == kKinds - 1;
  if (values) {
    float c1 = 1.f, c2 = 0.f;
    if (p.vr_coef) { c1 = p.vr_coef[0]; c2 = p.vr_coef[1]; }
    load_vmix<D>(p, x, b, g, j0, c1, c2, lane);
    stage_plain<D>(x, tile, lane);
  } else {
    load_tile<D>(x, row_ptr<float>(p.k, b, g, 0), p.k.stride_s, j0, p.Sk, lane);
    const f32x4v one = {1.f, 1.f, 1.f, 1.f};
    stage_norm<D, true, true>(p, x, one, p.rope_k_pos0 + j0, p.Sk - 1 - j0, tile, lane);
  }
  wave_sync();
  char* const dst = (values ? m.v : kind == 0 ? m.k_rm : m.k_tr) + t * kTileBytes<D>;
  const bool small = tile_small<D>(x);
  if ((values || kind == 0) && lane == 0) (values ? m.v_small : m.k_small)[t] = small;
  if (kind == 1) emit_tr<D>(tile, dst, lane, small ? kPart : 1.f);  // forward: values, backward: keys
  else emit_rm<D>(tile, dst, lane, small ? kPart : 1.f);
}

// ---- forward, as fwd_f32_kernel
template <int D>
__global__ __launch_bounds__(kThreads, 2) void fwd_split_kernel(KArgs a) {
  const segpt_attn_params& p = a.p;
  using T = T32<D>;
  // in the loop Qhat's units (and before it one fp32 tile behind them), after it the four waves' results
  __shared__ __attribute__((aligned(16))) char lds[std::max(kTileBytes<D> + 4 * T::kTile, 4 * kWaves * T::kTile)];
  char* const qs = lds;
  float* const tiles = reinterpret_cast<float*>(lds);
  __shared__ float msm[kWaves][32], lsm[kWaves][32];
  const int tid = threadIdx.x, lane = tid & 63;
  const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
  const int ln = lane & 31, hh = lane >> 5;
  const int n_qt = tiles_of(p.Sq), rep = p.H / p.Hkv;
  const Item item = split_item(blockIdx.x, n_qt, p.B * p.Hkv, rep, 2 * (int64_t)tiles_of(p.Sk) * kTileBytes<D>);
  const int b = item.pair / p.Hkv, g = item.pair % p.Hkv, h = g * rep + item.member;
  const int qt = n_qt - 1 - item.tile, q0 = qt * kRows;
  int kend = p.Sk;
  if (p.causal) kend = min(p.Sk, q0 + kRows + p.q_start);
  const int n_kt = tiles_of(kend);
  const SplitMap m = split_map<D>(a, false);
  const int64_t kv0 = ((int64_t)b * p.Hkv + g) * tiles_of(p.Sk), first = kv0 * kTileBytes<D>;
  const char *ktiles = m.k_rm + first, *vtiles = m.v + first;
  const uint32_t *k_small = m.k_small + kv0, *v_small = m.v_small + kv0;
  // step i of a tile uses half i of its keys, then of its values; requested kAhead steps before
  constexpr int MB = T::kMB, kSteps = 2 * MB, kAhead = D == 64 ? 3 : MB == 1 ? 1 : 2;
  Half half[kSteps];
  auto source = [&](int jt, int i) {
    return (i < MB ? ktiles : vtiles) + (int64_t)jt * kTileBytes<D> + i % MB * kHalfBytes;
  };
  const uint32_t flags = first_flags(k_small, n_kt, lane) | first_flags(v_small, n_kt, lane);
  if (wave < n_kt) {
#pragma unroll
    for (int i = 0; i < kAhead; ++i) half[i] = load_half(source(wave, i), lane);
  }
  bool q_small;
  {
    f32x4v qraw[T::kPasses], gs;
    load_tile<D>(qraw, row_ptr<float>(p.q, b, h, 0), p.q.stride_s, q0, p.Sq, lane);
#pragma unroll
    for (int e = 0; e < 4; ++e) gs[e] = gprod<D>(p, 4 * (lane % T::kLPR) + e) * p.sm_scale * kLog2e;
    float* const tile = reinterpret_cast<float*>(lds + kTileBytes<D>);  // every wave writes the same values
    stage_norm<D, true, true>(p, qraw, gs, p.rope_q_pos0 + q0, p.Sq - 1 - q0, tile, lane);
    wave_sync();
    q_small = tile_small<D>(qraw);
    emit_rm<D>(tile, qs, lane, q_small ? kPart : 1.f, wave, kWaves);
  }
  __syncthreads();

  f32x16 o[T::kMB];
#pragma unroll
  for (int mb = 0; mb < T::kMB; ++mb) o[mb] = zero16();
  float mrow = -INFINITY, l = 0.f;  // l: this lane's half of the keys
  const int qlim = p.causal ? min(q0 + ln + p.q_start, p.Sk - 1) : p.Sk - 1;  // last visible key
  const int n_full = p.causal ? min(p.Sk, q0 + p.q_start + 1) / kRows : p.Sk / kRows;  // tiles that need no mask

  // S^T of a tile: mask, maximum, probabilities
  auto softmax = [&](int jt, f32x16& s) {
    if (jt >= n_full) {
#pragma unroll
      for (int r = 0; r < 16; ++r)
        if (jt * kRows + crow(r, hh) > qlim) s[r] = -INFINITY;
    }
    float mx = s[0];
#pragma unroll
    for (int r = 1; r < 16; ++r) mx = fmaxf(mx, s[r]);
    mx = fmaxf(mrow, half_max(mx));
    const float mu = mx == -INFINITY ? 0.f : mx;
    if (any_lane(mx > mrow)) {  // some row has a new maximum
      const float corr = __builtin_amdgcn_exp2f(mrow - mu);
      l *= corr;
#pragma unroll
      for (int mb = 0; mb < T::kMB; ++mb)
#pragma unroll
        for (int r = 0; r < 16; ++r) o[mb][r] *= corr;
      mrow = mx;
    }
    float part[2] = {0.f, 0.f};
#pragma unroll
    for (int r = 0; r < 16; ++r) {
      s[r] = __builtin_amdgcn_exp2f(s[r] - mu);
      part[r & 1] += s[r];
    }
    l += part[0] + part[1];
  };
  const bool small = any_small(flags, k_small, n_kt, lane) | any_small(0, v_small, n_kt, lane) | q_small;
  int jt = wave;
#pragma unroll 1
  for (; !small && jt < n_kt; jt += kWaves) {
    const int next = jt + kWaves < n_kt ? jt + kWaves : jt;  // past the end: this tile's once more, unused
    auto request = [&](int i) { half[i % kSteps] = load_half(i < kSteps ? source(jt, i) : source(next, i - kSteps), lane); };
    Dot dot;
#pragma unroll
    for (int i = 0; i < MB; ++i) {
      request(i + kAhead);
      dot.add(half[i], qs + i * kHalfBytes, lane);
      step_end();
    }
    f32x16 s = dot.sum();
    softmax(jt, s);
    const Scores3 probs = split16<false>(s, 1.f);
#pragma unroll
    for (int i = MB; i < kSteps; ++i) {
      step_end();
      request(i + kAhead);
      add_tr(half[i], probs, o[i - MB]);
    }
    step_end();
  }
#pragma unroll 1
  for (; jt < n_kt; jt += kWaves) {  // some tile has small values
    const bool ks = k_small[jt], vs = v_small[jt];
    Dot dot;
    dot.add_scaled<D>(source(jt, 0), ks, qs, q_small, lane);
    f32x16 s = dot.sum();
    softmax(jt, s);
    const Scores3 probs = split16<false>(s, kPart);
#pragma unroll
    for (int i = MB; i < kSteps; ++i) {
      step_end();
      add_tr_scaled(load_half(source(jt, i), lane), vs, probs, o[i - MB]);
    }
  }

  const float lt = half_sum(l);
  if (hh == 0) { msm[wave][ln] = mrow; lsm[wave][ln] = lt; }
  __syncthreads();  // nobody reads Qhat any more
  put_rows<D>(tiles + wave * T::kTile, o, lane);
  __syncthreads();
  merge_waves<D>(p, b, h, q0, msm, lsm, tiles, T::kTile, tid);
}

// the rm units of a workgroup's stationary rows into LDS
template <int D>
__device__ __forceinline__ void fetch_units(char* lds, const char* tile, int tid) {
#pragma unroll
  for (int i = 0; i < kTileBytes<D>; i += 16 * kThreads)
    if (kTileBytes<D> % (16 * kThreads) == 0 || i + 16 * tid < kTileBytes<D>)
      *reinterpret_cast<u32x4*>(lds + i + 16 * tid) = *reinterpret_cast<const u32x4*>(tile + i + 16 * tid);
}

// ---- dQ: S^T and dP^T (lane = query), T^T += Khat^T dS^T
// `lds` holds in the loop the units of Qhat and dO (of Khat and V' below), after it the four waves' results
template <int D>
constexpr int kBwdLds = std::max(2 * kTileBytes<D>, 4 * kWaves * T32<D>::kTile);
template <int D>
constexpr int kBwdRed = kWaves * std::max(D, 64);
template <int D>
__device__ __forceinline__ void bwd_dq_split(const KArgs& a, int block, char* lds, float* red) {
  const segpt_attn_params& p = a.p;
  using T = T32<D>;
  char *const qs = lds, *const ds = lds + kTileBytes<D>;
  float* const tiles = reinterpret_cast<float*>(lds);
  const int tid = threadIdx.x, lane = tid & 63;
  const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
  const int ln = lane & 31, hh = lane >> 5;
  const int n_qt = tiles_of(p.Sq), rep = p.H / p.Hkv;
  const Item item = split_item(block, n_qt, p.B * p.Hkv, rep, 3 * (int64_t)tiles_of(p.Sk) * kTileBytes<D>);
  const int b = item.pair / p.Hkv, g = item.pair % p.Hkv, h = g * rep + item.member;
  const int qt = n_qt - 1 - item.tile, q0 = qt * kRows;
  int kend = p.Sk;
  if (p.causal) kend = min(p.Sk, q0 + kRows + p.q_start);
  const int n_kt = tiles_of(kend);
  const SplitMap m = split_map<D>(a, true);
  const int64_t kv0 = ((int64_t)b * p.Hkv + g) * tiles_of(p.Sk), first = kv0 * kTileBytes<D>, mine = ((int64_t)b * p.H + h) * n_qt + qt;
  const uint32_t *k_small = m.k_small + kv0, *v_small = m.v_small + kv0;
  const bool q_small = m.q_small[mine], d_small = m.d_small[mine];
  const char *ktiles = m.k_rm + first, *vtiles = m.v + first, *kttiles = m.k_tr + first;
  // step i of a tile: half i of the keys (scores), of the values (dP), of the keys again (T)
  constexpr int MB = T::kMB, kSteps = 3 * MB, kAhead = MB == 1 ? 2 : 3;
  Half half[kSteps];
  auto source = [&](int jt, int i) {
    return (i < MB ? ktiles : i < 2 * MB ? vtiles : kttiles) + (int64_t)jt * kTileBytes<D> + i % MB * kHalfBytes;
  };
  const uint32_t flags = first_flags(k_small, n_kt, lane) | first_flags(v_small, n_kt, lane);
  if (wave < n_kt) {
#pragma unroll
    for (int i = 0; i < kAhead; ++i) half[i] = load_half(source(wave, i), lane);
  }
  fetch_units<D>(qs, m.q_rm + mine * kTileBytes<D>, tid);
  fetch_units<D>(ds, m.d_rm + mine * kTileBytes<D>, tid);
  const float lse = m.stat[mine * 64 + ln], delta = m.stat[mine * 64 + 32 + ln];
  __syncthreads();
  f32x16 t[T::kMB];
#pragma unroll
  for (int mb = 0; mb < T::kMB; ++mb) t[mb] = zero16();
  const int qlim = p.causal ? min(q0 + ln + p.q_start, p.Sk - 1) : p.Sk - 1;
  const int n_full = p.causal ? min(p.Sk, q0 + p.q_start + 1) / kRows : p.Sk / kRows;

  // dS^T of a tile
  auto gradient = [&](int jt, f32x16& s, const f32x16& dp) {
#pragma unroll
    for (int r = 0; r < 16; ++r) s[r] = prob(s[r], lse);
    if (jt >= n_full) {
#pragma unroll
      for (int r = 0; r < 16; ++r)
        if (jt * kRows + crow(r, hh) > qlim) s[r] = 0.f;
    }
#pragma unroll
    for (int r = 0; r < 16; ++r) s[r] *= dp[r] - delta;
  };
  const bool small = any_small(flags, k_small, n_kt, lane) | any_small(0, v_small, n_kt, lane) | q_small | d_small;
  int jt = wave;
#pragma unroll 1
  for (; !small && jt < n_kt; jt += kWaves) {
    const int next = jt + kWaves < n_kt ? jt + kWaves : jt;
    auto request = [&](int i) { half[i % kSteps] = load_half(i < kSteps ? source(jt, i) : source(next, i - kSteps), lane); };
    Dot dot[2];
#pragma unroll
    for (int i = 0; i < 2 * MB; ++i) {
      request(i + kAhead);
      dot[i / MB].add(half[i], (i < MB ? qs : ds) + i % MB * kHalfBytes, lane);
      step_end();
    }
    f32x16 s = dot[0].sum();
    gradient(jt, s, dot[1].sum());
    const LaneScores grads = split_lanes<true>(s);
#pragma unroll
    for (int i = 2 * MB; i < kSteps; ++i) {
      step_end();
      request(i + kAhead);
      add_tr(half[i], grads.s, t[i - 2 * MB], grads.f);
    }
    step_end();
  }
#pragma unroll 1
  for (; jt < n_kt; jt += kWaves) {  // some tile has small values
    const bool kf = k_small[jt], vf = v_small[jt];
    Dot dot[2];
    dot[0].add_scaled<D>(source(jt, 0), kf, qs, q_small, lane);
    dot[1].add_scaled<D>(source(jt, MB), vf, ds, d_small, lane);
    f32x16 s = dot[0].sum();
    gradient(jt, s, dot[1].sum());
    const Scores3 grads = split16<true>(s, kPart);
#pragma unroll
    for (int i = 2 * MB; i < kSteps; ++i) {
      step_end();
      add_tr_scaled(load_half(source(jt, i), lane), kf, grads, t[i - 2 * MB]);
    }
  }

  __syncthreads();
  put_rows<D>(tiles + wave * T::kTile, t, lane);
  __syncthreads();
  finish_dq<D>(a, b, h, q0, (int)mine, tiles, T::kTile, red, tid);
}

// ---- dK, dV of one kv head: S = Qhat Khat^T and dP = dO V'^T (lane = key), dV^T += dO^T P, dK^T += Qhat^T dS.  The query tiles
// that see the keys, of all query heads of the group one after the other, are dealt out to 4 f32_parts waves; a workgroup
// leaves one part of the sum (bwd_dkdv_f32_kernel leaves one per query head and share: twice the traffic at two heads a group).
template <int D>
__device__ __forceinline__ void bwd_dkdv_split(const KArgs& a, int block, char* lds, float* stat_lds) {
  const segpt_attn_params& p = a.p;
  using T = T32<D>;
  char *const ks = lds, *const vs = lds + kTileBytes<D>;
  float* const tiles = reinterpret_cast<float*>(lds);
  float(*const stat)[64] = reinterpret_cast<float(*)[64]>(stat_lds);
  const int tid = threadIdx.x, lane = tid & 63;
  const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
  const int ln = lane & 31, hh = lane >> 5;
  const Item item = split_item(block, tiles_of(p.Sk), p.B * p.Hkv, a.f32_parts, 4 * (int64_t)(p.H / p.Hkv) * tiles_of(p.Sq) * kTileBytes<D>);  // the first key tiles are the heaviest
  const int kt_i = item.tile, part_i = item.member, bg = item.pair;
  const int b = bg / p.Hkv, g = bg % p.Hkv, rep = p.H / p.Hkv;
  const int j0 = kt_i * kRows;
  const SplitMap m = split_map<D>(a, true);
  const int n_qt = tiles_of(p.Sq);
  const int first = p.causal ? max(0, j0 - p.q_start) / kRows : 0;  // the first tile that holds a query seeing key j0
  const int step = kWaves * a.f32_parts;
  const bool k_small = m.k_small[(int64_t)bg * tiles_of(p.Sk) + kt_i], v_small = m.v_small[(int64_t)bg * tiles_of(p.Sk) + kt_i];
  const int64_t mine = ((int64_t)bg * tiles_of(p.Sk) + kt_i) * kTileBytes<D>, head = (int64_t)(b * p.H + g * rep) * n_qt;
  const char *qrm = m.q_rm + head * kTileBytes<D>, *qtr = m.q_tr + head * kTileBytes<D>;
  const char *drm = m.d_rm + head * kTileBytes<D>, *dtr = m.d_tr + head * kTileBytes<D>;
  const float* stats = m.stat + head * 64;
  const uint32_t *q_small = m.q_small + head, *d_small = m.d_small + head;
  int it = first + part_i * kWaves + wave, left = rep;  // tile within its head, query heads still to come with this one
  auto settle = [&](int& tile, int& heads) {  // tiles past a head's last one are the next head's first visible ones
    while (tile >= n_qt && heads > 0) { tile -= n_qt - first; --heads; }
  };
  if (first < n_qt) settle(it, left);
  else left = 0;
  // step i of a tile: half i of the queries (scores), of dO (dP), of dO again (dV), of the queries again (dK)
  constexpr int MB = T::kMB, kSteps = 4 * MB, kAhead = 3;
  Half half[kSteps];
  auto source = [&](int tile, int i) {
    return (i < MB ? qrm : i < 2 * MB ? drm : i < 3 * MB ? dtr : qtr) + (int64_t)tile * kTileBytes<D> + i % MB * kHalfBytes;
  };
  float st = 0.f;
  const uint32_t flags = first_flags(q_small, rep * n_qt, lane) | first_flags(d_small, rep * n_qt, lane);
  int at = (rep - left) * n_qt + it;  // tile within the group
  if (left > 0) {
#pragma unroll
    for (int i = 0; i < kAhead; ++i) half[i] = load_half(source(at, i), lane);
    st = stats[(int64_t)at * 64 + lane];
  }
  fetch_units<D>(ks, m.k_rm + mine, tid);
  fetch_units<D>(vs, m.v + mine, tid);
  __syncthreads();
  f32x16 dk[T::kMB], dv[T::kMB];
#pragma unroll
  for (int mb = 0; mb < T::kMB; ++mb) dk[mb] = dv[mb] = zero16();

  // S and dP of a tile to P and dS
  auto probabilities = [&](int i0, f32x16& s) {
#pragma unroll
    for (int q = 0; q < 4; ++q) {
      const f32x4v ls = *reinterpret_cast<const f32x4v*>(&stat[wave][8 * q + 4 * hh]);
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
  };
  auto gradients = [&](f32x16& s, const f32x16& dp) {
#pragma unroll
    for (int q = 0; q < 4; ++q) {
      const f32x4v de = *reinterpret_cast<const f32x4v*>(&stat[wave][32 + 8 * q + 4 * hh]);
#pragma unroll
      for (int e = 0; e < 4; ++e) s[4 * q + e] *= dp[4 * q + e] - de[e];
    }
  };
  const bool small = any_small(flags, q_small, rep * n_qt, lane) | any_small(0, d_small, rep * n_qt, lane) | k_small | v_small;
#pragma unroll 1
  while (left > 0 && !small) {
    int next_it = it + step, next_left = left;
    settle(next_it, next_left);
    const int next = next_left > 0 ? (rep - next_left) * n_qt + next_it : at;
    auto request = [&](int i) { half[i % kSteps] = load_half(i < kSteps ? source(at, i) : source(next, i - kSteps), lane); };
    stat[wave][lane] = st;
    st = stats[(int64_t)next * 64 + lane];
    wave_sync();
    Dot dot[2];
#pragma unroll
    for (int i = 0; i < 2 * MB; ++i) {
      request(i + kAhead);
      dot[i / MB].add(half[i], (i < MB ? ks : vs) + i % MB * kHalfBytes, lane);
      step_end();
    }
    f32x16 s = dot[0].sum();
    const f32x16 dp = dot[1].sum();
    probabilities(it * kRows, s);
    const LaneScores probs = split_lanes<false>(s);
    gradients(s, dp);
    const LaneScores grads = split_lanes<true>(s);
#pragma unroll
    for (int i = 2 * MB; i < kSteps; ++i) {
      step_end();
      request(i + kAhead);
      if (i < 3 * MB) add_tr(half[i], probs.s, dv[i - 2 * MB], probs.f);
      else add_tr(half[i], grads.s, dk[i - 3 * MB], grads.f);
    }
    step_end();
    wave_sync();
    it = next_it;
    left = next_left;
    at = next;
  }
#pragma unroll 1
  while (left > 0) {  // some tile has small values
    const bool qf = q_small[at], df = d_small[at];
    wave_sync();
    stat[wave][lane] = stats[(int64_t)at * 64 + lane];
    wave_sync();
    Dot dot[2];
    dot[0].add_scaled<D>(source(at, 0), qf, ks, k_small, lane);
    dot[1].add_scaled<D>(source(at, MB), df, vs, v_small, lane);
    f32x16 s = dot[0].sum();
    probabilities(it * kRows, s);
    const Scores3 probs = split16<false>(s, kPart);
#pragma unroll
    for (int i = 2 * MB; i < 3 * MB; ++i) {
      step_end();
      add_tr_scaled(load_half(source(at, i), lane), df, probs, dv[i - 2 * MB]);
    }
    gradients(s, dot[1].sum());
    const Scores3 grads = split16<true>(s, kPart);
#pragma unroll
    for (int i = 3 * MB; i < kSteps; ++i) {
      step_end();
      add_tr_scaled(load_half(source(at, i), lane), qf, grads, dk[i - 3 * MB]);
    }
    it += step;
    settle(it, left);
    at = (rep - left) * n_qt + it;
  }

  const int part = tid % T::kLPR;
  const int64_t out = ((int64_t)bg * a.f32_parts + part_i) * p.Sk * D;
  auto leave = [&](const f32x16 (&acc)[T::kMB], float* to) {
    __syncthreads();
    put_rows<D>(tiles + wave * T::kTile, acc, lane);
    __syncthreads();
#pragma unroll
    for (int row = tid / T::kLPR; row < kRows; row += kThreads / T::kLPR)
      if (j0 + row < p.Sk)
        *reinterpret_cast<f32x4v*>(to + out + (int64_t)(j0 + row) * D + 4 * part) = sum_waves<D>(tiles, T::kTile, row, part);
  };
  leave(dk, a.f32_dk_part);
  leave(dv, a.f32_dv_part);
}

template <int D>
__global__ __launch_bounds__(kThreads, 2) void bwd_dq_split_kernel(KArgs a) {
  __shared__ __attribute__((aligned(16))) char lds[kBwdLds<D>];
  __shared__ __attribute__((aligned(16))) float red[kBwdRed<D>];
  bwd_dq_split<D>(a, blockIdx.x, lds, red);
}
// On its own the dK/dV launch's first workgroup adds up the scale gradient behind the others' back: in the finish kernel it was the longest one (finish
// 6.9 -> 4.7 us at 512 rows, 109 -> 24 at 9216; the other seven of the first kXcds workgroups keep the rest on their XCDs).
template <int D>
__global__ __launch_bounds__(kThreads, (D == 128 ? 1 : 2)) void bwd_dkdv_split_kernel(KArgs a) {
  __shared__ __attribute__((aligned(16))) char lds[kBwdLds<D>];
  __shared__ __attribute__((aligned(16))) float stat[kBwdRed<D>];
  if (blockIdx.x < kXcds) {
    float* const sums = reinterpret_cast<float*>(lds);
    if (blockIdx.x == 0) reduce_scale_grad<kThreads>(a, threadIdx.x, sums, sums + kThreads);
    return;
  }
  bwd_dkdv_split<D>(a, blockIdx.x - kXcds, lds, stat);
}
// Both, dK/dV first: they need the pre-pass and not each other, so the heavy dQ workgroups fill the causal tail of dK/dV and a launch is saved; the
// finish kernel adds up the scale gradient.  For grids of one or two resident rounds each, where the tail counts (f32_split_both).  Backward, us, two
// launches -> one: 2 x 8 / 4 heads of 64, 1000 tokens 75.5 -> 76.3, 400 tokens 41.7 -> 38.8; 1 x 4 heads, 700 tokens 43.2 -> 39.1; 4 x 8
// heads, 1000 tokens (1024 dQ workgroups) 143.3 -> 142.7; 3 x 6 / 2 heads of 32, 1000 tokens 56.5 -> 53.8.  And where what dQ streams stays in the
// L2 beside what dK/dV does (32 / 4 heads, 256 queries, 8192 keys 361 -> 410; 16 / 2 heads, 2048 tokens 223 -> 255; 32 / 1 heads, 900 tokens 147 -> 137).  head_dim 128 has its own register
// bound for dK/dV; larger grids want a pair's tiles pinned to an XCD and have the longer sum of the scale gradient.
template <int D>
__global__ __launch_bounds__(kThreads, 2) void bwd_both_split_kernel(KArgs a, int n_dkdv) {
  __shared__ __attribute__((aligned(16))) char lds[kBwdLds<D>];
  __shared__ __attribute__((aligned(16))) float red[kBwdRed<D>];
  if ((int)blockIdx.x < n_dkdv) bwd_dkdv_split<D>(a, blockIdx.x, lds, red);
  else bwd_dq_split<D>(a, blockIdx.x - n_dkdv, lds, red);
}

int n_tiles(int n) { return (n + kRows - 1) / kRows; }

dim3 split_grid(int tiles, int pairs, int members, int extra = 0) {
  return dim3((unsigned)(extra + (int64_t)tiles * pairs * members));
}

template <int D>
int launch_prep(const KArgs& a, bool bwd, hipStream_t st) {
  const segpt_attn_params& p = a.p;
  const int64_t kv = (int64_t)p.B * p.Hkv * n_tiles(p.Sk), q = (int64_t)p.B * p.H * n_tiles(p.Sq);
  const int64_t jobs = bwd ? 4 * q + 3 * kv : 2 * kv;
  const dim3 grid((unsigned)((jobs + kWaves - 1) / kWaves)), block(kThreads);
  if (bwd) hipLaunchKernelGGL((split_prep_kernel<D, true>), grid, block, 0, st, a);
  else hipLaunchKernelGGL((split_prep_kernel<D, false>), grid, block, 0, st, a);
  return (int)hipGetLastError();
}
template <int D>
int launch_attn(const KArgs& a, hipStream_t st) {
  hipLaunchKernelGGL(fwd_split_kernel<D>, split_grid(n_tiles(a.p.Sq), a.p.B * a.p.Hkv, a.p.H / a.p.Hkv), dim3(kThreads), 0, st, a);
  return (int)hipGetLastError();
}
template <int D>
int launch_dq(const KArgs& a, hipStream_t st) {
  hipLaunchKernelGGL(bwd_dq_split_kernel<D>, split_grid(n_tiles(a.p.Sq), a.p.B * a.p.Hkv, a.p.H / a.p.Hkv), dim3(kThreads), 0, st, a);
  return (int)hipGetLastError();
}
template <int D>
int launch_dkdv(const KArgs& a, hipStream_t st) {
  const segpt_attn_params& p = a.p;
  hipLaunchKernelGGL(bwd_dkdv_split_kernel<D>, split_grid(n_tiles(p.Sk), p.B * p.Hkv, a.f32_parts, kXcds), dim3(kThreads), 0, st, a);
  const int rc = (int)hipGetLastError();
  return rc ? rc : launch_finish_f32(a, st);
}

}  // namespace

// Parts of dK and dV per kv head: one resident round of 512 workgroups, every wave with a tile; never more than the
// workspace of the other kernels has, one per query head and f32_dkdv_splits.
int f32_split_parts(const segpt_attn_params& p) {
  const int units = n_tiles(p.Sk) * p.B * p.Hkv, rep = p.H / p.Hkv;
  int want = (kResident + units - 1) / units;
  const int most = (rep * n_tiles(p.Sq) + kWaves - 1) / kWaves;
  // Less than two rounds of workgroups that all walk more than an L2 holds: the heaviest of them alone take as long as the rest, so two parts each.
  // Backward, us, one part -> two (fp32 instructions): 12 / 3 heads of 64, 8192 tokens 3241 -> 2432 (3135); 20 / 5 heads, 4096 tokens 1223 -> 1050 (1361);
  // 32 / 4 heads of 128, 4096 tokens 4364 -> 2991 (5247).  One head a group walks less: 5 heads, 4096 tokens 293 -> 296.
  const bool walks = stream_per_xcd(p.B * p.Hkv, 4 * (int64_t)rep * n_tiles(p.Sq) * p.D * (kUnitBytes / 16)) > kStreamLimit;
  if (want == 1 && units <= 2 * kResident && walks && rep > 1) want = 2;
  return std::max(1, std::min({want, most, rep * f32_dkdv_splits(p)}));
}
// Where splitting pays.  The pre-pass is a launch more (4 to 7 us, 12 for a backward of 16 heads of 1000 tokens) and 6 bytes an
// element written and read again, so a key has to be used by several workgroups (`users`) and a wave has to have a few tiles.  The fp32 instructions'
// times go in steps, rounds of 256 or 512 resident workgroups of `n_kt` tiles; hence lines in n_kt and in workgroups (`grid`).  Us of a call, plain
// operands, fp32 instructions -> here; two heads a group where no other is given:
//   forward  128, 4 heads:  128 tokens 13.4 -> 18.2, 192 19.7 -> 20.8, 1000 59.7 -> 36.8;  16 heads: 192 19.9 -> 21.4, 512 34.5 -> 28.3
//            one head a group:  8 heads: 256 20.5 -> 21.6, 320 26.6 -> 24.1;  16: 256 20.5 -> 23.2, 320 26.6 -> 25.8;  32: 256 20.9 -> 26.2, 320 27.4 -> 30.2, 400 46 -> 35;
//            64: 256 34.3 -> 31.4;  four a group:  32: 256 20.9 -> 22.3, 320 27.3 -> 26.4;  8 x 32 / 4 heads, one query, 4096 keys 227 -> 156
//            64, 16 heads:  256 10.9 -> 13.6, 384 14.5 -> 15.5, 512 17.8 -> 17.0, 1000 32.6 -> 26.2;  32 heads: 512 20.4 -> 19.8, 768 40 -> 33; 144 heads of 2048 842 -> 505
//            one head a group:  8 heads: 512 17.7 -> 16.7;  12: 512 17.6 -> 19.2, 600 20.9 -> 21.4;  16: 512 17.7 -> 18.3, 600 22.3 -> 21.4;  17: 512 19.3 -> 21.5
//            32, 12 heads:  512 11.1 -> 12.7, 768 15.6 -> 15.4;  24: 512 12.1 -> 13.9;  48 heads: 256 8.6 -> 11.5, 384 13.6 -> 13.4
//            one head a group:  24: 640 14.4 -> 16.6;  48: 448 15.9 -> 16.5, 480 18.8 -> 17.8;  80: 448 24.0 -> 25.2;  128: 256 16.6 -> 18.8, 384 27 -> 28, 448 35 -> 32;
//            256: 320 41 -> 36;  four a group:  256: 160 18.1 -> 17.5
//   backward 128:  4 heads: 64 tokens 48 -> 33, 1000 153 -> 81;  16 heads: 128 49 -> 38, 512 125 -> 73;  one query: 4 heads, 2048 keys 180 -> 89, 8 x 32 / 4
//            heads, 4096 keys 2730 -> 605;  32 x 16 heads, one key 86 -> 66
//            64, 16 heads:  256 34 -> 29, 384 48 -> 38, 1000 110 -> 76;  32 heads: 192 39 -> 32, 384 65 -> 44
//            32, 12 heads:  384 29 -> 26, 512 34 -> 32, 768 55 -> 40;  48 heads: 192 31 -> 29, 384 54 -> 40;  one head a group, 128: 128 28 -> 31, 256 57 -> 56
// One or two kv heads whose dK/dV workgroups each walk all queries of very many tiles, backward: the streams outgrow every cache
//   64, one kv head:  16 heads of 4096 tokens (2048 users) 1097 -> 998, 12 of 6000 (2256) 1737 -> 1811, 16 of 6000 2275 -> 2350, 32 of 4096 2157 -> 2180;  two: 32 of 8192 8252 -> 8585
//   32, one kv head:  64 heads of 4096 tokens (8192) 2342 -> 2245, of 8192 8979 -> 9150
bool f32_split_pays(const segpt_attn_params& p, bool bwd) {
  const int n_qt = n_tiles(p.Sq), n_kt = n_tiles(p.Sk), rep = p.H / p.Hkv;
  const int64_t heads = (int64_t)p.B * p.H, pairs = heads * n_qt * n_kt, grid = heads * n_qt;
  const int64_t users = (int64_t)rep * n_qt;  // workgroups that read a key tile
  if (users < 8 && !(bwd && p.D == 128)) return false;  // one query against a long cache: split keys used once or twice
  if (bwd && p.D <= 64 && p.B * p.Hkv <= 2 && users > (p.D == 64 ? 2200 : 12000)) return false;
  if (p.D == 128) return bwd || n_kt >= 13 || (n_kt >= 10 && (grid <= 192 || users >= 24)) || (n_kt >= 6 && grid >= 512);
  if (p.D == 64) return bwd ? n_kt >= 12 : n_kt >= 24 || (n_kt >= 16 && heads <= 16 && (heads <= 8 || n_kt >= 19 || users >= 32));
  if (bwd) return pairs >= 3072;
  return pairs >= 5000 && (n_kt >= 24 || (n_kt >= 15 && grid > 512) || (n_kt >= 14 && grid >= 1792) || grid >= 2560 || (rep >= 4 && users >= 14 && grid > 512));
}
size_t f32_split_bytes(const segpt_attn_params& p, bool bwd) {
  if (!f32_split_pays(p, bwd)) return 0;
  const size_t tile = (size_t)p.D * (kUnitBytes / 16), kv = (size_t)p.B * p.Hkv * n_tiles(p.Sk), q = (size_t)p.B * p.H * n_tiles(p.Sq);
  return (bwd ? (3 * kv + 4 * q) * tile + q * (64 * sizeof(float) + 2 * sizeof(uint32_t)) : 2 * kv * tile) + kv * 2 * sizeof(uint32_t);
}

int launch_split_prep(const KArgs& a, bool bwd, hipStream_t st) {
  switch (a.p.D) {
    case 32: return launch_prep<32>(a, bwd, st);
    case 64: return launch_prep<64>(a, bwd, st);
    case 128: return launch_prep<128>(a, bwd, st);
    default: return (int)hipErrorInvalidValue;
  }
}
int launch_fwd_split(const KArgs& a, hipStream_t st) {
  switch (a.p.D) {
    case 32: return launch_attn<32>(a, st);
    case 64: return launch_attn<64>(a, st);
    case 128: return launch_attn<128>(a, st);
    default: return (int)hipErrorInvalidValue;
  }
}
int launch_bwd_dq_split(const KArgs& a, hipStream_t st) {
  switch (a.p.D) {
    case 32: return launch_dq<32>(a, st);
    case 64: return launch_dq<64>(a, st);
    case 128: return launch_dq<128>(a, st);
    default: return (int)hipErrorInvalidValue;
  }
}
bool f32_split_both(const KArgs& a) {
  const segpt_attn_params& p = a.p;
  return p.D != 128 && n_tiles(p.Sq) * (int64_t)p.B * p.H <= kPinnedGrid && n_tiles(p.Sk) * (int64_t)p.B * p.Hkv * a.f32_parts <= kPinnedGrid &&
         stream_per_xcd(p.B * p.Hkv, 3 * (int64_t)n_tiles(p.Sk) * p.D * (kUnitBytes / 16)) <= kL2Bytes;
}
int launch_bwd_both_split(const KArgs& a, hipStream_t st) {
  const segpt_attn_params& p = a.p;
  const int n_dkdv = n_tiles(p.Sk) * p.B * p.Hkv * a.f32_parts, n_dq = n_tiles(p.Sq) * p.B * p.H;
  const dim3 grid((unsigned)(n_dkdv + n_dq)), block(kThreads);
  switch (p.D) {
    case 32: hipLaunchKernelGGL(bwd_both_split_kernel<32>, grid, block, 0, st, a, n_dkdv); break;
    case 64: hipLaunchKernelGGL(bwd_both_split_kernel<64>, grid, block, 0, st, a, n_dkdv); break;
    default: return (int)hipErrorInvalidValue;
  }
  return (int)hipGetLastError();
}
int launch_bwd_dkdv_split(const KArgs& a, hipStream_t st) {
  switch (a.p.D) {
    case 32: return launch_dkdv<32>(a, st);
    case 64: return launch_dkdv<64>(a, st);
    case 128: return launch_dkdv<128>(a, st);
    default: return (int)hipErrorInvalidValue;
  }
}

}  // namespace segpt
