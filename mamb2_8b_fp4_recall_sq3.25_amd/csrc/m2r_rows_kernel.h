// Multi-token scan of the quantized codecs with each state row spread over
// one to eight lanes, for gfx950: the packed 52-byte rows (legacy, stored-scale
// tiers, ridge latent) and the dense 3-bit rows.
//
//   legacy  mamba2_recall/state_codec.py:105-176 (_sq_scan)
//   tier    scripts/state_ppl_codec_v10.py:78-154 (_tier_scan)
//   ridge   scripts/fp4_zero_predictor_codec_v1.py:76-236 (_latent_scan, scan)
//   dense3  mamba2_recall/state_codec_dense3.py:82-148 (_scan)
//
// A token's chain is: update every carried coordinate, the tier's maximum,
// its scale, the codes; the next token starts from codes * scale.  Its length
// is what bounds a scan of few rows, and vector issue one of many, so here
//  - a wave holds 64 / LPR rows of LPR lanes, a lane the coordinates of 8 /
//    LPR halves of readout segments (m2r_step.h), each in one tier: the
//    tier's maximum and the readout are DPP steps, with no barrier and no LDS
//    exchange between waves.  With eight lanes a batch-1 layer is 1,024
//    waves, one per SIMD;
//  - the codes stay in registers, as integers in binary32, from token to
//    token: no packing and unpacking (a third of the one-lane step's vector
//    work), the nibble planes taken apart and put together once per call;
//  - tokens come in blocks of 16: the next block's inputs are loaded into
//    registers while this one steps, and a token reads its operands from LDS
//    (eight lanes: one token ahead).  dt activations are evaluated 64 tokens
//    at a time.
// 512 tokens of a batch-1 layer, against the several waves per 64-row slot
// and (dense rows) one lane per row before: ridge 24/44/60 629 -> 328 us
// (the records kernel included), tier 32/32/64 596 -> 264, legacy 651 -> 270,
// dense3 2,049 -> 337.
// The arithmetic is that of m2r_step.h and m2r_dense3.hip: codes and scales
// equal a call per token bit for bit, and so does a ridge row's y, whose
// one-token step sums in the same order (the other codecs' y differ from it
// by the order of a binary32 sum).
#pragma once
#include "m2r_rows.h"
#include "m2r_step.h"

namespace m2r {

// Geometry of rows on LPR lanes: lane j holds the LANE_HALVES consecutive
// halves from half j * LANE_HALVES on, half m of a lane in SLOTS(m) register
// slots from OFF(m) on (the widest of the lanes' halves m).
template <int N8, int N4, int MODE, int LPR>
struct RowGeom {
  static constexpr bool D3 = MODE == MODE_DENSE3;
  static constexpr int NL = D3 ? 128 : N8 + N4, HALVES = 8 / LPR;
  static constexpr int pos(int j) { return D3 ? 16 * j : half_pos(N8, N4, j); }
  static constexpr int at[9] = {pos(0), pos(1), pos(2), pos(3), pos(4), pos(5), pos(6), pos(7), pos(8)};
  static constexpr int size(int h) { return at[h + 1] - at[h]; }
  static constexpr bool first(int h) { return at[h] < (D3 ? 64 : N8); }   // half h lies in the first tier
  static constexpr int widest(int m) {
    int w = 0;
    for (int j = 0; j < LPR; ++j) w = size(j * HALVES + m) > w ? size(j * HALVES + m) : w;
    return w;
  }
  static constexpr int narrowest(int m) {
    int w = NL;
    for (int j = 0; j < LPR; ++j) w = size(j * HALVES + m) < w ? size(j * HALVES + m) : w;
    return w;
  }
  static constexpr int sum_to(int m) { return m == 0 ? 0 : sum_to(m - 1) + widest(m - 1); }
  template <int M>
  struct Half {   // half m of every lane
    static constexpr int SLOTS = widest(M), MIN = narrowest(M), OFF = sum_to(M);
    static constexpr int count_first() {
      int n = 0;
      for (int j = 0; j < LPR; ++j) n += first(j * HALVES + M) ? 1 : 0;
      return n;
    }
    static constexpr bool ALL8 = count_first() == LPR, NONE8 = count_first() == 0;
  };
  static constexpr int K = sum_to(HALVES);   // slots of a lane
  static constexpr bool pure() {             // every lane's halves lie in one tier
    for (int j = 0; j < LPR; ++j)
      for (int m = 1; m < HALVES; ++m)
        if (first(j * HALVES + m) != first(j * HALVES)) return false;
    return true;
  }
  static constexpr bool PURE = pure();
  static constexpr int lane4() {   // the first lane with a half of the second tier
    int h = 0;
    while (first(h)) ++h;
    return h / HALVES;
  }
  static constexpr int LANE4 = lane4();
  // register slot of internal position p within its lane, or of its lane's row of slots
  static constexpr int slot(int p) {
    int h = 0;
    while (p >= at[h + 1]) ++h;
    return (h / HALVES) * K + sum_to(h % HALVES) + p - at[h];
  }
  static_assert(K % 4 == 0, "whole chunks");
};

constexpr int ROWS_TOKENS = 16;    // tokens of a block

template <int N8, int N4, int MODE, int LPR>
struct RowsSmem {
  using Geo = RowGeom<N8, N4, MODE, LPR>;
  static constexpr int K = Geo::K, T = ROWS_TOKENS, RW = 64 / LPR, ROWS = 4 * RW;
  static constexpr bool RIDGE = MODE == MODE_RIDGE;
  // per token: readout weights and b, lane-major (K per lane, zero past a
  // half's coordinates), then the sum of b.c and a flag that a b is not
  // finite, and the ridge codec's latent corrections and dead-tier dot
  // products (as in its record)
  static constexpr int O_B = LPR * K, O_SUM = 2 * LPR * K, O_LAT = O_SUM + 4, O_TREE = O_LAT + 4;
  static constexpr int FLOATS = O_SUM + (RIDGE ? 12 : 4);
  struct Tokens {
    alignas(16) float tok[T][FLOATS];
    alignas(16) uint16_t x[T][ROWS];
    alignas(16) uint16_t y[T][ROWS + 8];                           // + a column for lanes without a readout
    alignas(16) uint16_t raw[RIDGE ? 1 : T][2][RIDGE ? 8 : 128];   // b and c rows before the table's gather
  };
  union {
    Tokens t;
    uint8_t code[MODE == MODE_DENSE3 ? 1 : ROWS][Geo::NL];   // after the last token
  };
  alignas(16) f32x4 act[4][64];   // dt, decay, range flag of 64 tokens, per wave (its head)
};

// A flag as the magnitude that a range test rejects.
constexpr float ROWS_BAD = 0x1p127f;

template <int CTRL>
__device__ __forceinline__ float dpp_move(float v) {
  return __builtin_bit_cast(float, __builtin_amdgcn_update_dpp(0, __builtin_bit_cast(int, v), CTRL, 0xF, 0xF, true));
}
// Maximum of non-negative values over a row's aligned LPR lanes (quad
// permutes, then the half-row mirror of quads that hold one value each), as
// integers, which order them alike and need no canonical operands.
template <int LPR>
__device__ __forceinline__ float row_max(float v) {
  uint32_t m = __builtin_bit_cast(uint32_t, v);
  if constexpr (LPR > 1) m = max(m, __builtin_bit_cast(uint32_t, dpp_move<0xB1>(__builtin_bit_cast(float, m))));
  if constexpr (LPR > 2) m = max(m, __builtin_bit_cast(uint32_t, dpp_move<0x4E>(__builtin_bit_cast(float, m))));
  if constexpr (LPR > 4) m = max(m, __builtin_bit_cast(uint32_t, dpp_move<0x141>(__builtin_bit_cast(float, m))));
  return __builtin_bit_cast(float, m);
}

// f(integral_constant<int, 0>) ... f(integral_constant<int, N - 1>)
template <int N, int I = 0, class F>
__device__ __forceinline__ void static_for(F&& f) {
  if constexpr (I < N) {
    f(std::integral_constant<int, I>{});
    static_for<N, I + 1>(f);
  }
}

// RN(1/d) up to half an ulp plus 2^-46, for a positive normal d: enough for
// the two-sided quantizer (its bracket leaves 2^-24 of slack), which keeps
// no code the exact quotient could differ in.
__device__ __forceinline__ float recip_near(float d) {
  const float y = __builtin_amdgcn_rcpf(d);
  return __builtin_fmaf(__builtin_fmaf(-d, y, 1.0f), y, y);
}

template <int N8, int N4, int NZ, int MODE, int LPR>
__global__ __launch_bounds__(256) __attribute__((amdgpu_waves_per_eu(LPR == 8 || LPR == 4 ? 3 : 2, 8)))
void k_rows_scan(StepArgs a, int equalizer, int wg_heads, int tokens) {
  using Geo = RowGeom<N8, N4, MODE, LPR>;
  using Smem = RowsSmem<N8, N4, MODE, LPR>;
  constexpr bool RIDGE = MODE == MODE_RIDGE, D3 = MODE == MODE_DENSE3, DEN32 = MODE == MODE_LEGACY || D3;
  constexpr int K = Geo::K, T = ROWS_TOKENS, NL = Geo::NL, W8 = N8 / 2, W4 = N4 / 2, HALVES = Geo::HALVES;
  constexpr int RW = Smem::RW, ROWS = Smem::ROWS;
  constexpr bool PURE = Geo::PURE;
  constexpr int SETS = PURE ? 1 : 2;            // tiers of a lane (its own, or both)
  constexpr int NLAT = LPR == 1 ? 2 : 1;        // latent coefficients of a lane (by its parity, or both)
  __shared__ Smem sm;
  const int tid = threadIdx.x, lane = tid & 63;
  const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
  const int b = blockIdx.z;
  // the first L of a batch row's a.L tokens (a ridge scan's records: these alone)
  const int H = a.H, P = a.P, G = a.G, L = RIDGE ? tokens : a.L;
  // a wave's rows: RW consecutive p of one head; the four waves take
  // consecutive blocks of wg_heads heads of one group
  const int wave_blocks = 4 / wg_heads;
  const int h0 = blockIdx.y * wg_heads;
  const int g = h0 / (H / G);
  auto head_of = [&](int w) { return h0 + w / wave_blocks; };
  auto p_of = [&](int w) { return (blockIdx.x * wave_blocks + w % wave_blocks) * RW; };
  const int h = head_of(wave), p0 = p_of(wave);
  const int part = lane % LPR;
  const int r = RW * wave + lane / LPR;         // workgroup row
  const bool valid = p0 + lane / LPR < P;       // (P % 8 == 0)
  const size_t row = (size_t)(b * H + h) * P + p0 + lane / LPR;
  const float av = a.A[h], Dh = load_param(a.D, a.d_f32, h), bias = load_param(a.dt_bias, a.db_f32, h);

  // per half of the lane: its first internal position, its coordinates and its tier
  int start[HALVES], count[HALVES];
  bool first[HALVES];
  static_for<HALVES>([&](auto mc) __attribute__((always_inline)) {
    constexpr int M = decltype(mc)::value;
    using Half = typename Geo::template Half<M>;
    start[M] = count[M] = 0;
    first[M] = Half::ALL8;
    static_for<LPR>([&](auto jc) __attribute__((always_inline)) {
      constexpr int J = decltype(jc)::value, S = Geo::at[J * HALVES + M], E = Geo::at[J * HALVES + M + 1];
      constexpr bool F8 = Geo::first(J * HALVES + M);
      start[M] = part == J ? S : start[M];
      count[M] = Half::SLOTS == Half::MIN ? Half::SLOTS : (part == J ? E - S : count[M]);
      if constexpr (!Half::ALL8 && !Half::NONE8) first[M] = part == J ? F8 : first[M];
    });
  });
  // the constants of a lane's tiers
  float lim[SETS], rlim[SETS], top_lim[SETS];
#pragma unroll
  for (int e = 0; e < SETS; ++e) {
    const bool t8 = PURE ? first[0] : e == 0;
    lim[e] = D3 ? 3.0f : (t8 ? 127.0f : 7.0f);
    rlim[e] = D3 ? 1.0f / 3.0f : (t8 ? 1.0f / 127.0f : 1.0f / 7.0f);
    top_lim[e] = D3 ? QTOP3 : (t8 ? QTOP127 : QTOP7);
  }

  // ---- block inputs: into registers (load_block), then LDS (stage_block)
  constexpr int PIECES = RIDGE ? T / 4 : T / 8, XPIECES = (T * ROWS / 8 + 255) / 256;
  u32x4 piece[PIECES] = {}, xpiece[XPIECES] = {};
  // ridge: 16-byte piece `lane` of the records of tokens wave + 4 k, written
  // where its chunk of coordinates (or its scalars) goes
  int rec_dst = -1;
  if constexpr (RIDGE) {
    const int f = 4 * lane;
    static_for<NL / 4>([&](auto cc) __attribute__((always_inline)) {
      constexpr int C = 4 * decltype(cc)::value, SLOT = Geo::slot(C);
      rec_dst = f == REC_CW + C ? SLOT : rec_dst;
      rec_dst = f == REC_B + C ? Smem::O_B + SLOT : rec_dst;
    });
    rec_dst = f == REC_CW + NL ? Smem::O_LAT : rec_dst;
    rec_dst = f == REC_TREE ? Smem::O_TREE : rec_dst;
    rec_dst = f == REC_SBC ? Smem::O_SUM : rec_dst;
  }
  // else: piece tid % 32 (b: 0-15, c: 16-31) of the raw rows of tokens tid / 32 + 8 k
  const int rp = tid & 31, rt = tid >> 5;
  const uint16_t* raw_src = (rp < 16 ? a.Bm : a.Cm) + 8 * (rp & 15);
  // x and y: piece i of 8 rows of a token, tid + 256 k over (token, piece)
  auto xy_row = [&](int i, int t, size_t& at) {   // false: past P
    const int w = i / (RW / 8), p = p_of(w) + 8 * (i % (RW / 8));
    at = ((size_t)(b * a.L + t) * H + head_of(w)) * P + p;
    return p < P;
  };
  auto load_block = [&](int t0) {   // (past the last token: stale values, never stepped)
    if constexpr (RIDGE) {
#pragma unroll
      for (int k = 0; k < PIECES; ++k) {
        const int t = t0 + wave + 4 * k;
        if (t < L) piece[k] = ((const u32x4*)(a.rec + ((size_t)(b * L + t) * G + g) * REC_FLOATS))[lane];
      }
    } else {
#pragma unroll
      for (int k = 0; k < PIECES; ++k) {
        const int t = t0 + rt + 8 * k;
        if (t < L) piece[k] = *(const u32x4*)(raw_src + ((size_t)(b * a.L + t) * G + g) * 128);
      }
    }
#pragma unroll
    for (int k = 0; k < XPIECES; ++k) {
      const int e = tid + 256 * k, t = e / (ROWS / 8);
      size_t at;
      if (t < T && t0 + t < L && xy_row(e % (ROWS / 8), t0 + t, at)) xpiece[k] = *(const u32x4*)(a.x + at);
    }
  };
  // the table's gather: lane l prepares packed positions (dense rows:
  // coordinates) l and l + 64 of tokens wave + 4 k
  int gpos[2] = {0, 0}, gdst[2] = {-1, -1};
  float wf[2] = {1.f, 1.f}, rf[2] = {1.f, 1.f};
  if constexpr (!RIDGE) {
#pragma unroll
    for (int e = 0; e < 2; ++e) {
      const int n = lane + 64 * e;
      const uint32_t tb = a.perm[g * 128 + (D3 ? n : packed_lane<N8, N4>(n))];
      gpos[e] = (int)(tb & 127u);   // in-bounds for any table
      if (D3 && equalizer) {
        const int k = (int)(int8_t)tb;
        gpos[e] = n;
        wf[e] = __builtin_ldexpf(1.0f, -k);   // exp2(-k), exact
        rf[e] = __builtin_ldexpf(1.0f, k);
      }
      static_for<NL / 4>([&](auto cc) __attribute__((always_inline)) {
        constexpr int C = 4 * decltype(cc)::value, SLOT = Geo::slot(C);
        gdst[e] = (n & ~3) == C ? SLOT + (n & 3) : gdst[e];
      });
    }
  }
  auto stage_block = [&]() {
#pragma unroll
    for (int k = 0; k < XPIECES; ++k) {
      const int e = tid + 256 * k;
      if (e < T * ROWS / 8) *(u32x4*)&sm.t.x[e / (ROWS / 8)][8 * (e % (ROWS / 8))] = xpiece[k];
    }
    if constexpr (RIDGE) {
#pragma unroll
      for (int k = 0; k < PIECES; ++k) {
        u32x4 v = piece[k];
        if (rec_dst == Smem::O_SUM)   // the record says that every b is finite
          v.y = v.y == 0u ? __builtin_bit_cast(uint32_t, ROWS_BAD) : 0u;
        if (rec_dst >= 0) *(u32x4*)&sm.t.tok[wave + 4 * k][rec_dst] = v;
      }
    } else {
#pragma unroll
      for (int k = 0; k < PIECES; ++k) *(u32x4*)&sm.t.raw[rt + 8 * k][rp >> 4][8 * (rp & 15)] = piece[k];
      __syncthreads();   // the raw rows are in LDS
#pragma unroll
      for (int k = 0; k < T / 4; ++k) {
        const int t = wave + 4 * k;
        float bv[2], cv[2];
#pragma unroll
        for (int e = 0; e < 2; ++e) {
          bv[e] = h2f(sm.t.raw[t][0][gpos[e]]) * wf[e];
          cv[e] = h2f(sm.t.raw[t][1][gpos[e]]) * rf[e];
          if (gdst[e] >= 0) {
            sm.t.tok[t][gdst[e]] = cv[e];
            sm.t.tok[t][Smem::O_B + gdst[e]] = bv[e];
          }
        }
        const bool bad = !(__builtin_fabsf(bv[0]) < 0x1p30f && __builtin_fabsf(bv[1]) < 0x1p30f);
        const float sum = D3 ? 0.f : wave_sum(bv[0] * cv[0] + bv[1] * cv[1]);
        const bool any_bad = __builtin_amdgcn_ballot_w64(bad) != 0;
        if (lane == 0) *(float2*)&sm.t.tok[t][Smem::O_SUM] = make_float2(sum, any_bad ? ROWS_BAD : 0.f);
      }
    }
  };

  load_block(0);
  // ---- the lane's codes (as integers in binary32), scales and latents
  float q[K], s[SETS];
#pragma unroll
  for (int i = 0; i < K; ++i) q[i] = 0.f;
#pragma unroll
  for (int e = 0; e < SETS; ++e) s[e] = 0.f;
  float z[NLAT], ls[NLAT], rls[NLAT];
  uint32_t zbyte[NLAT];
#pragma unroll
  for (int e = 0; e < NLAT; ++e) {
    zbyte[e] = 0;
    z[e] = 0.f;
    ls[e] = RIDGE ? h2f(a.lscale[2 * g + (NLAT == 2 ? e : lane & 1)]) : 1.f;
    rls[e] = recip_half(ls[e]);
  }
  if (valid) {
#pragma unroll
    for (int e = 0; e < SETS; ++e) {
      const bool t8 = PURE ? first[0] : e == 0;
      s[e] = h2f(D3 ? a.s8[row * 2 + (t8 ? 0 : 1)] : (t8 ? a.s8 : a.s4)[row]);
    }
    static_for<HALVES>([&](auto mc) __attribute__((always_inline)) {
      constexpr int M = decltype(mc)::value;
      using Half = typename Geo::template Half<M>;
      if constexpr (D3) {   // 16 coordinates: two bytes of each plane
        uint32_t pl[3];
#pragma unroll
        for (int k = 0; k < 3; ++k) pl[k] = *(const uint16_t*)(a.lo + row * 48 + 16 * k + start[M] / 8);
#pragma unroll
        for (int i = 0; i < Half::SLOTS; ++i) {
          const int u = (int)(((pl[0] >> i) & 1u) | (((pl[1] >> i) & 1u) << 1) | (((pl[2] >> i) & 1u) << 2));
          q[Half::OFF + i] = (float)(u >= 4 ? u - 8 : u);
        }
      } else {
        const bool t8 = first[M];
        const int tstart = t8 ? start[M] : start[M] - N8, TW = t8 ? N8 : N4, W = t8 ? W8 : W4;
#pragma unroll
        for (int c = 0; c < Half::SLOTS / 4; ++c) {
          if (4 * c < count[M]) {
            // chunk c: four nibbles of plane word `w` (even or odd packed
            // lanes), or all four of a tier's last half word
            const int tp = tstart + 4 * c, w = tp >> 3;
            const bool last4 = 8 * w + 8 > TW;
            const size_t o = row * W + 4 * w;
            const uint16_t* pa = (const uint16_t*)((t8 ? a.lo : a.q4) + o);
            const uint32_t wa = (uint32_t)pa[0] | (last4 ? 0u : (uint32_t)pa[1] << 16);
            uint32_t wb = 0u;
            if (t8) {
              const uint16_t* pb = (const uint16_t*)(a.hi + o);
              wb = (uint32_t)pb[0] | (last4 ? 0u : (uint32_t)pb[1] << 16);
            }
#pragma unroll
            for (int m = 0; m < 4; ++m) {
              const int sh = last4 ? 8 * (m & 1) + 4 * (m >> 1) : 8 * m + ((tp >> 2) & 1) * 4;
              const int lo4 = (int)((wa >> sh) & 15u), hi4 = (int)((wb >> sh) & 15u);
              const int u8 = (hi4 << 4) | lo4;
              q[Half::OFF + 4 * c + m] = (float)(t8 ? (u8 > 127 ? u8 - 256 : u8) : (lo4 > 7 ? lo4 - 16 : lo4));
            }
          }
        }
      }
    });
    if constexpr (RIDGE) {
#pragma unroll
      for (int e = 0; e < NLAT; ++e) {
        zbyte[e] = a.latent[row * 2 + (NLAT == 2 ? e : lane & 1)];
        z[e] = e4m3_byte_to_f32<0>(zbyte[e]) * ls[e];
      }
    }
  }
  // zeros past the halves' coordinates
  for (int i = tid; i < T * Smem::FLOATS; i += 256) (&sm.t.tok[0][0])[i] = 0.f;
  __syncthreads();
  stage_block();

  // a token's operands; few lanes per row (many slots): w and b are read where they are used
  constexpr bool AHEAD = LPR == 8;
  struct Operands {
    f32x4 w[AHEAD ? K / 4 : 1], b[AHEAD ? K / 4 : 1], act;
    float2 sum;
    float lat[2], tree_c[2], tree_b[2];
    uint16_t x;
  };
  const int ycol = part == 0 ? r : ROWS;
  for (int t0 = 0; t0 < L; t0 += T) {
    const int n = min(T, L - t0);
    // (dt, decay) of tokens t0 .. t0 + 63, one per lane: a one-head
    // workgroup's waves take turns, else each wave does its own head's
    if ((t0 & 63) == 0 && (wg_heads > 1 || wave == ((t0 >> 6) & 3))) {
      const int t = min(t0 + lane, L - 1);
      const float2 v = dt_activation<false>(h2f(a.dt[(size_t)(b * a.L + t) * H + h]) + bias, av);
      // |b| < 2^30 (2^16 without an equalizer), |dt| < 2^60 and |decay| <
      // 2^100 keep every update of finite operands finite
      const bool bounded = __builtin_fabsf(v.x) < 0x1p60f && __builtin_fabsf(v.y) < 0x1p100f;
      sm.act[wg_heads > 1 ? wave : 0][lane] = f32x4{v.x, v.y, bounded ? 0.f : ROWS_BAD, 0.f};
    }
    if (t0 + T < L) load_block(t0 + T);
    __syncthreads();   // the block is staged

    const f32x4* act = sm.act[wg_heads > 1 ? wave : 0];
    auto operands = [&](int i) __attribute__((always_inline)) {
      Operands o;
      const float* tk = sm.t.tok[i];
      if constexpr (AHEAD) {
#pragma unroll
        for (int c = 0; c < K / 4; ++c) {
          o.w[c] = *(const f32x4*)(tk + part * K + 4 * c);
          o.b[c] = *(const f32x4*)(tk + Smem::O_B + part * K + 4 * c);
        }
      }
      o.sum = *(const float2*)(tk + Smem::O_SUM);
      o.act = act[(t0 & 63) + i];
      if constexpr (RIDGE) {
#pragma unroll
        for (int e = 0; e < NLAT; ++e) {
          const int k = NLAT == 2 ? e : lane & 1;
          o.lat[e] = tk[Smem::O_LAT + k];
          o.tree_c[e] = tk[Smem::O_TREE + k];
          o.tree_b[e] = tk[Smem::O_TREE + 2 + k];
        }
      }
      o.x = sm.t.x[i][r];
      return o;
    };
    auto step = [&](const Operands& o, int i) __attribute__((always_inline)) {
      const float dtv = o.act.x, decay = o.act.y, x = h2f(o.x);
      const float* tk = sm.t.tok[i];
      bool finite_in = __builtin_fmaxf(o.sum.y, o.act.z) < ROWS_BAD && __builtin_fabsf(x) <= 65504.f;
#pragma unroll
      for (int e = 0; e < SETS; ++e) finite_in = finite_in && __builtin_fabsf(s[e]) <= 65504.f;
      // readout, update and maximum, half by half
      float v[K], chain[HALVES], amax[SETS];
#pragma unroll
      for (int e = 0; e < SETS; ++e) amax[e] = 0.f;
      static_for<HALVES>([&](auto mc) __attribute__((always_inline)) {
        constexpr int M = decltype(mc)::value;
        using Half = typename Geo::template Half<M>;
        const float sh = PURE ? s[0] : (first[M] ? s[0] : s[SETS - 1]);
        float racc = 0.f, rend = 0.f, hmax = 0.f;
        float rsum[4] = {0.f, 0.f, 0.f, 0.f};   // (dense rows: four chains)
#pragma unroll
        for (int c = 0; c < Half::SLOTS / 4; ++c) {
          const int k0 = Half::OFF + 4 * c;
          f32x4 w4, b4;
          if constexpr (AHEAD) {
            w4 = o.w[k0 / 4];
            b4 = o.b[k0 / 4];
          } else {
            w4 = *(const f32x4*)(tk + part * K + k0);
            b4 = *(const f32x4*)(tk + Smem::O_B + part * K + k0);
          }
#pragma unroll
          for (int e = 0; e < 4; ++e) {
            const float prior = q[k0 + e] * sh;   // exact
            const float bdt = b4[e] * dtv;
            float u = state_update(prior, decay, bdt * x);
            // (many slots: the update is formed here, and its operands die)
            if constexpr (!AHEAD) asm volatile("" : "+v"(u));
            v[k0 + e] = u;
            // the dense rows read the update out, the packed rows (as their
            // one-token step) the prior, completed below
            if constexpr (D3) rsum[e] = __builtin_fmaf(u, w4[e], rsum[e]);
            else racc = __builtin_fmaf(prior, w4[e], racc);
          }
          hmax = max3_abs(hmax, v[k0], v[k0 + 1]);
          hmax = max3_abs(hmax, v[k0 + 2], v[k0 + 3]);
          // (past a half's coordinates the code is 0, but 0 times an infinite
          // scale is not: a shorter half's chain ends here)
          if (4 * c + 4 < Half::SLOTS && 4 * c + 4 >= Half::MIN) rend = count[M] == 4 * c + 4 ? racc : rend;
        }
        if constexpr (D3) chain[M] = (rsum[0] + rsum[1]) + (rsum[2] + rsum[3]);
        else chain[M] = Half::SLOTS == Half::MIN ? racc : (count[M] == Half::SLOTS ? racc : rend);
        if constexpr (PURE) {
          amax[0] = max3_abs(amax[0], hmax, 0.f);
        } else if constexpr (Half::ALL8 || Half::NONE8) {
          amax[Half::ALL8 ? 0 : SETS - 1] = max3_abs(amax[Half::ALL8 ? 0 : SETS - 1], hmax, 0.f);
        } else {
          amax[0] = max3_abs(amax[0], first[M] ? hmax : 0.f, 0.f);
          amax[SETS - 1] = max3_abs(amax[SETS - 1], first[M] ? 0.f : hmax, 0.f);
        }
      });
      // the tiers' maxima over the row's lanes
      float den[SETS], stored[SETS];
      if constexpr (PURE) {
        const float m0 = row_max<LPR>(first[0] ? amax[0] : 0.f), m1 = row_max<LPR>(first[0] ? 0.f : amax[0]);
        amax[0] = first[0] ? m0 : m1;
      } else {
#pragma unroll
        for (int e = 0; e < SETS; ++e) amax[e] = row_max<LPR>(amax[e]);
      }
#pragma unroll
      for (int e = 0; e < SETS; ++e) {
        den[e] = requant_den(amax[e], lim[e], rlim[e]);
        stored[e] = round_to_half(den[e]);
      }

      // readout: the segments' left fold, on the row's first lane
      {
        float acc;
        if constexpr (LPR == 8) {
          const float seg = chain[0] + dpp_move<0xB1>(chain[0]);
          acc = seg + dpp_move<0x102>(seg);   // row_shl 2, 4, 6
          acc = acc + dpp_move<0x104>(seg);
          acc = acc + dpp_move<0x106>(seg);
        } else if constexpr (LPR == 4) {
          const float seg = chain[0] + chain[1];
          acc = seg + dpp_move<0x55>(seg);   // quad lanes 1, 2, 3
          acc = acc + dpp_move<0xAA>(seg);
          acc = acc + dpp_move<0xFF>(seg);
        } else if constexpr (LPR == 2) {
          const float s0 = chain[0] + chain[1], s1 = chain[2] + chain[3];
          acc = s0 + s1;
          acc = acc + dpp_move<0xB1>(s0);
          acc = acc + dpp_move<0xB1>(s1);
        } else {
          acc = (((chain[0] + chain[1]) + (chain[2] + chain[3])) + (chain[4] + chain[5])) + (chain[6] + chain[7]);
        }
        float out;
        if constexpr (D3) {
          out = acc + x * Dh;
        } else {
          if constexpr (RIDGE) {   // + z0 dot0 + z1 dot1
            const float zd = z[0] * (o.tree_c[0] + o.lat[0]);
            if constexpr (NLAT == 2) acc = acc + zd + z[NLAT - 1] * (o.tree_c[NLAT - 1] + o.lat[NLAT - 1]);
            else acc = acc + zd + dpp_move<0xB1>(zd);
          }
          out = decay * acc + x * (dtv * o.sum.x + Dh);
        }
        sm.t.y[i][ycol] = f2h(out);
      }
      if constexpr (RIDGE) {   // latent step (bit-exact), as in m2r_step.h
#pragma unroll
        for (int e = 0; e < NLAT; ++e) {
          const float zn = state_update(z[e], decay, (x * dtv) * o.tree_b[e]);
          const float lq = __builtin_fminf(__builtin_fmaxf(latent_quotient(zn, ls[e], rls[e]), -448.f), 448.f);
          zbyte[e] = f32x2_to_e4m3(lq, lq) & 0xFFu;   // clamped, never NaN
          z[e] = __builtin_amdgcn_cvt_f32_fp8((int)zbyte[e], 0) * ls[e];
        }
      }
      // new codes (tier_requant of m2r_step.h, d3_half of m2r_dense3.hip)
      bool unclamped = finite_in, zero[SETS];
#pragma unroll
      for (int e = 0; e < SETS; ++e) {
        zero[e] = !DEN32 && stored[e] == 0.f;
        // (2^-14 to 65504, as one comparison of integers; an overflowed scale
        // has no reciprocal for the two-sided quantizer)
        const bool normal = __builtin_bit_cast(uint32_t, stored[e]) - 0x38800000u <= 0x477FE000u - 0x38800000u;
        unclamped = unclamped && (DEN32 || zero[e] || normal);
      }
      if (__builtin_amdgcn_ballot_w64(!unclamped) == 0) {
        float yh[SETS], yl[SETS];
#pragma unroll
        for (int e = 0; e < SETS; ++e) {
          const float y = zero[e] ? 0.f : recip_near(DEN32 ? den[e] : stored[e]);
          yh[e] = __builtin_fmaf(y, TWO_SIDED_REL, y);
          yl[e] = __builtin_fmaf(y, -TWO_SIDED_REL, y);
        }
        uint32_t diff = 0u;
        static_for<HALVES>([&](auto mc) __attribute__((always_inline)) {
          constexpr int M = decltype(mc)::value;
          using Half = typename Geo::template Half<M>;
          const float yhm = PURE ? yh[0] : (first[M] ? yh[0] : yh[SETS - 1]);
          const float ylm = PURE ? yl[0] : (first[M] ? yl[0] : yl[SETS - 1]);
#pragma unroll
          for (int k = Half::OFF; k < Half::OFF + Half::SLOTS; ++k) {
            const uint32_t th = two_sided_code(v[k], yhm, ylm, 0.0f, diff);
            asm volatile("" : "+v"(diff));   // one three-input bitwise operation per coordinate
            q[k] = __builtin_bit_cast(float, th) - 0x1.8p23f;
          }
        });
        if (__builtin_amdgcn_ballot_w64(diff != 0u) != 0) {   // near a half-integer: exact quotients
          float d[SETS], ry[SETS];
#pragma unroll
          for (int e = 0; e < SETS; ++e) {
            d[e] = zero[e] ? 1.f : (DEN32 ? den[e] : stored[e]);
            ry[e] = zero[e] ? 0.f : 1.0f / d[e];
          }
          static_for<HALVES>([&](auto mc) __attribute__((always_inline)) {
            constexpr int M = decltype(mc)::value;
            using Half = typename Geo::template Half<M>;
            const int e = PURE ? 0 : (first[M] ? 0 : SETS - 1);
            const float dm = e == 0 ? d[0] : d[SETS - 1], rm = e == 0 ? ry[0] : ry[SETS - 1];
#pragma unroll
            for (int k = Half::OFF; k < Half::OFF + Half::SLOTS; ++k) {
              q[k] = (float)quantize_code_unclamped(v[k], dm, rm);
              if constexpr (!AHEAD) asm volatile("" : "+v"(q[k]));
            }
          });
        }
      } else {
        // not finite, or a binary16-subnormal or infinite stored scale: clamped
        // exact quotients (a zero, infinite or NaN divisor divides through d = 1, y = 0)
        float d[SETS], ry[SETS], top[SETS];
#pragma unroll
        for (int e = 0; e < SETS; ++e) {
          const float by = DEN32 ? den[e] : stored[e];
          const bool none = !(by > 0.f) || by == __builtin_inff();
          d[e] = none ? 1.f : by;
          ry[e] = none ? 0.f : 1.0f / d[e];
          top[e] = DEN32 || stored[e] > 0.f ? top_lim[e] : 0.f;
        }
        static_for<HALVES>([&](auto mc) __attribute__((always_inline)) {
          constexpr int M = decltype(mc)::value;
          using Half = typename Geo::template Half<M>;
          const int e = PURE ? 0 : (first[M] ? 0 : SETS - 1);
          const float dm = e == 0 ? d[0] : d[SETS - 1], rm = e == 0 ? ry[0] : ry[SETS - 1];
          const float tm = e == 0 ? top[0] : top[SETS - 1];
#pragma unroll
          for (int k = Half::OFF; k < Half::OFF + Half::SLOTS; ++k) {
            q[k] = k - Half::OFF < count[M] ? (float)quantize_code(v[k], dm, rm, tm) : 0.f;
            if constexpr (!AHEAD) asm volatile("" : "+v"(q[k]));
          }
        });
      }
#pragma unroll
      for (int e = 0; e < SETS; ++e) s[e] = stored[e];
    };
    if constexpr (AHEAD) {   // the operands of the next token are read while this one steps
      Operands o0 = operands(0);
      int i = 0;
      for (; i + 1 < n; i += 2) {
        const Operands o1 = operands(i + 1);
        step(o0, i);
        o0 = operands(min(i + 2, T - 1));
        step(o1, i + 1);
      }
      if (i < n) step(o0, i);
    } else {
      for (int i = 0; i < n; ++i) step(operands(i), i);
    }
    __syncthreads();   // every wave is past the block's operands; its readouts are in LDS
#pragma unroll
    for (int k = 0; k < XPIECES; ++k) {
      const int e = tid + 256 * k, t = e / (ROWS / 8), i = e % (ROWS / 8);
      size_t at;
      if (t < n && xy_row(i, t0 + t, at)) *(u32x4*)(a.y + at) = *(const u32x4*)&sm.t.y[t][8 * i];
    }
    if (t0 + T < L) stage_block();
  }

  // ---- the rows' codes, scales and latents
  if (valid) {
    if constexpr (PURE) {
      if (part == 0 || part == Geo::LANE4) {
        if (D3) a.s8[row * 2 + (first[0] ? 0 : 1)] = f2h(s[0]);
        else (first[0] ? a.s8 : a.s4)[row] = f2h(s[0]);
      }
    } else if (part == 0) {
      a.s8[D3 ? row * 2 : row] = f2h(s[0]);
      if (D3) a.s8[row * 2 + 1] = f2h(s[SETS - 1]);
      else a.s4[row] = f2h(s[SETS - 1]);
    }
    if constexpr (RIDGE) {
#pragma unroll
      for (int e = 0; e < NLAT; ++e)
        if (part < 2) a.latent[row * 2 + (NLAT == 2 ? e : part)] = (uint8_t)zbyte[e];
    }
  }
  if constexpr (D3) {
    if (valid) {
      static_for<HALVES>([&](auto mc) __attribute__((always_inline)) {
        constexpr int M = decltype(mc)::value;
        using Half = typename Geo::template Half<M>;
        uint32_t pl[3] = {0u, 0u, 0u};
#pragma unroll
        for (int i = 0; i < Half::SLOTS; ++i) {
          const uint32_t c = (uint32_t)(int)q[Half::OFF + i];
#pragma unroll
          for (int k = 0; k < 3; ++k) pl[k] |= ((c >> k) & 1u) << i;
        }
#pragma unroll
        for (int k = 0; k < 3; ++k) *(uint16_t*)(a.lo + row * 48 + 16 * k + start[M] / 8) = (uint16_t)pl[k];
      });
    }
  } else {
    __syncthreads();   // the last block's readouts have left LDS
    static_for<HALVES>([&](auto mc) __attribute__((always_inline)) {
      constexpr int M = decltype(mc)::value;
      using Half = typename Geo::template Half<M>;
#pragma unroll
      for (int i = 0; i < Half::SLOTS; ++i)
        if (i < count[M]) sm.code[r][start[M] + i] = (uint8_t)(int)q[Half::OFF + i];
    });
    wave_sync();   // a wave's rows are written out by its own lanes
    // packed lane n of a tier of TW coordinates -> internal position
    auto internal = [](int n, int TW) {
      const int w = n & ~7;
      return w + 8 > TW ? w + 2 * (n & 1) + ((n & 3) >> 1) : w + 4 * (n & 1) + ((n & 7) >> 1);
    };
    const size_t row0 = (size_t)(b * H + h) * P + p0;
    const int rows = min(RW, P - p0);   // may be negative
#pragma unroll 4
    for (int i = lane; i < RW * W8; i += 64) {
      const int rr = i / W8, nn = 2 * (i % W8);
      if (rr < rows) {
        const uint8_t* c = sm.code[RW * wave + rr];
        const uint32_t c0 = c[internal(nn, N8)], c1 = c[internal(nn + 1, N8)];
        a.lo[row0 * W8 + i] = (uint8_t)((c0 & 15u) | (c1 << 4));
        a.hi[row0 * W8 + i] = (uint8_t)((c0 >> 4) | (c1 & 0xF0u));
      }
    }
#pragma unroll 4
    for (int i = lane; i < RW * W4; i += 64) {
      const int rr = i / W4, nn = 2 * (i % W4);
      if (rr < rows) {
        const uint8_t* c = sm.code[RW * wave + rr] + N8;
        const uint32_t c0 = c[internal(nn, N4)], c1 = c[internal(nn + 1, N4)];
        a.q4[row0 * W4 + i] = (uint8_t)((c0 & 15u) | (c1 << 4));
      }
    }
  }
}

template <int N8, int N4, int NZ, int MODE, int LPR>
inline hipError_t launch_rows_lanes(const StepArgs& a, int equalizer, int tokens, hipStream_t stream) {
  const int blocks = rows_blocks(LPR, a.P), heads = rows_heads(blocks, a.H / a.G);
  const dim3 grid((unsigned)((blocks * heads + 3) / 4), (unsigned)(a.H / heads), (unsigned)a.B);
  hipLaunchKernelGGL((k_rows_scan<N8, N4, NZ, MODE, LPR>), grid, dim3(256), 0, stream, a, equalizer, heads,
                     tokens);
  return hipGetLastError();
}

template <int N8, int N4, int NZ, int MODE>
inline hipError_t launch_rows_scan(const StepArgs& a, int equalizer, int tokens, hipStream_t stream) {
  constexpr int NL = MODE == MODE_DENSE3 ? 128 : N8 + N4;
  const int lanes = rows_lanes(NL, rows_slots(a.B, a.H, a.P));
  if (lanes == 8) return launch_rows_lanes<N8, N4, NZ, MODE, 8>(a, equalizer, tokens, stream);
  if (lanes == 4) return launch_rows_lanes<N8, N4, NZ, MODE, 4>(a, equalizer, tokens, stream);
  if (lanes == 2) return launch_rows_lanes<N8, N4, NZ, MODE, 2>(a, equalizer, tokens, stream);
  if constexpr (NL <= 72) return launch_rows_lanes<N8, N4, NZ, MODE, 1>(a, equalizer, tokens, stream);
  return hipErrorInvalidValue;   // (rows_lanes never asks for one lane there)
}

}  // namespace m2r
