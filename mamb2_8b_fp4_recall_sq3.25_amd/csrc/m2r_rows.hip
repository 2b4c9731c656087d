// Multi-token scans with each state row spread over several lanes, for gfx950.
//
//   s16     mamba2_recall/state_codec.py:65-102 (_s16_scan)
//   dense3, tier, legacy: m2r_rows_kernel.h
//
// Compiled with the max-ILP machine scheduler: 180 -> 167 us for 512 tokens
// of the FP16 carry at batch 1, against the default one.
#include "m2r_rows_kernel.h"
#include "m2r_rows.h"

namespace m2r {

// ---------------------------------------------------------------------------
// Multi-token scan with each row spread over eight lanes.
//
// With one lane per row (k_s16_step) a batch-1 layer is 128 waves, one on
// every eighth SIMD, each running 128 coordinates, a binary64 dt activation
// and two barriers per token: a serial chain, whatever the memory system
// does.  The carry's coordinates do not depend on each other (only the
// readout joins them), so here a wave holds 8 rows x 8 lanes of 16
// coordinates and a batch-1 layer is 1,024 waves, one per SIMD.
//  - The carry stays binary16 between tokens and enters the update through a
//    mixed-precision fma, as b and c do: 5 VALU instructions per coordinate
//    (RN(b dt), times x, update, readout, rounding), 6 with statistics.
//  - Tokens come in blocks of 32: b, c and x of the next block are loaded
//    into registers while this one steps and written to the other LDS
//    buffer at its end, so a token needs no barrier and waits only for LDS.
//    The readouts leave the same way, 64 contiguous bytes per token.
//  - The dt activation of 64 tokens is one lane-parallel evaluation of one
//    wave, the four waves taking turns.
// Per token of a 512-token call at batch 1 (8,192 rows): 0.27 us, with
// statistics 0.33, against 3.28 and 4.07 with one lane per row.
constexpr int S16_ROWS = 32;     // rows of a workgroup (four waves of 8)
constexpr int S16_TOKENS = 32;   // tokens of a block
constexpr int S16_K = 16;        // coordinates of a lane

struct S16RowsSmem {
  alignas(16) uint16_t bc[2][S16_TOKENS][2][128];   // b and c of the block's tokens, by block parity
  alignas(16) uint16_t x[2][S16_TOKENS][S16_ROWS];
  alignas(16) uint16_t y[S16_TOKENS][S16_ROWS];
  float2 act[64];                                   // (dt, decay) of 64 tokens
  float sub[4][2][128];                             // statistics: 4-row sub-tile sums of each wave
};

// v + the value of the lane 8 apart in its row of 16 lanes.
__device__ __forceinline__ float add_lane_xor8(float v) {
  const int iv = __builtin_bit_cast(int, v);
  return v + __builtin_bit_cast(float, __builtin_amdgcn_update_dpp(0, iv, 0x128, 0xF, 0xF, true));   // row_ror:8
}

template <bool STATS>
__global__ __launch_bounds__(256) void k_s16_rows(S16Args a) {
  __shared__ S16RowsSmem sm;
  constexpr int T = S16_TOKENS, K = S16_K;
  const int tid = threadIdx.x, lane = tid & 63;
  const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
  const int b = blockIdx.z, h = blockIdx.y;
  const int H = a.H, P = a.P, G = a.G, L = a.L;
  const int g = h / (H / G);
  const int pbase = blockIdx.x * S16_ROWS;
  const int nvalid = min(S16_ROWS, P - pbase);   // a multiple of 8: a wave's rows are all valid or none
  const int part = lane & 7;
  const int r = 8 * wave + (lane >> 3);          // workgroup row
  const bool valid = 8 * wave < nvalid;
  const float av = a.A[h], Dh = load_param(a.D, a.d_f32, h), bias = load_param(a.dt_bias, a.db_f32, h);

  // block loads: thread i takes 16-byte piece i % 32 (b: 0-15, c: 16-31) of
  // tokens i / 32 + 8 k, and threads below 128 piece i % 4 of x of token i / 4
  const int piece = tid & 31, tk = tid >> 5;
  const uint16_t* bc_src = (piece < 16 ? a.Bm : a.Cm) + 8 * (piece & 15);
  const int xt = tid >> 2, xp = 8 * (tid & 3);
  const bool xin = tid < 4 * T && xp < nvalid;
  u32x4 rbc[T / 8] = {}, rx = {};
  auto load_block = [&](int t0) {
#pragma unroll
    for (int k = 0; k < T / 8; ++k) {   // (past the last token: stale values, never stepped)
      const int t = t0 + tk + 8 * k;
      if (t < L) rbc[k] = *(const u32x4*)(bc_src + ((size_t)(b * L + t) * G + g) * 128);
    }
    if (xin && t0 + xt < L) rx = *(const u32x4*)(a.x + ((size_t)(b * L + t0 + xt) * H + h) * P + pbase + xp);
  };
  auto stage_block = [&](int buf) {
#pragma unroll
    for (int k = 0; k < T / 8; ++k) *(u32x4*)&sm.bc[buf][tk + 8 * k][piece >> 4][8 * (piece & 15)] = rbc[k];
    if (xin) *(u32x4*)&sm.x[buf][xt][xp] = rx;
  };

  load_block(0);
  _Float16 st[K];
  float sum[STATS ? K : 1];
  u32x4* const srow = (u32x4*)(a.state + ((size_t)(b * H + h) * P + pbase + r) * 128 + K * part);
  {
    const u32x4 v0 = valid ? srow[0] : u32x4{0u, 0u, 0u, 0u}, v1 = valid ? srow[1] : u32x4{0u, 0u, 0u, 0u};
#pragma unroll
    for (int i = 0; i < K; ++i)
      st[i] = __builtin_bit_cast(_Float16, (uint16_t)((i < 8 ? v0 : v1)[(i >> 1) & 3] >> (16 * (i & 1))));
  }
  if constexpr (STATS) {
#pragma unroll
    for (int i = 0; i < K; ++i) sum[i] = 0.f;
  }
  stage_block(0);
  const float mz = opaque_neg_zero();
  int buf = 0;
  for (int t0 = 0; t0 < L; t0 += T, buf ^= 1) {
    const int n = min(T, L - t0);
    if (t0 + T < L) load_block(t0 + T);
    if ((t0 & 63) == 0 && wave == ((t0 >> 6) & 3)) {   // (dt, decay) of tokens t0 .. t0 + 63, one per lane
      const int t = min(t0 + lane, L - 1);
      sm.act[lane] = dt_activation<true>(h2f(a.dt[(size_t)(b * L + t) * H + h]) + bias, av);
    }
    __syncthreads();   // the block's b, c and x are staged (and the previous block's readouts stored)
    struct Operands { u32x4 b0, b1, c0, c1; float2 act; uint16_t x; };
    auto operands = [&](int i) {
      const u32x4* pb = (const u32x4*)&sm.bc[buf][i][0][K * part];
      const u32x4* pc = (const u32x4*)&sm.bc[buf][i][1][K * part];
      return Operands{pb[0], pb[1], pc[0], pc[1], sm.act[(t0 & 63) + i], sm.x[buf][i][r]};
    };
    auto step = [&](const Operands& o, int i) {
      const float dtv = o.act.x, decay = o.act.y, x = h2f(o.x);
      float acc[2] = {0.f, 0.f};   // two readout chains
#pragma unroll
      for (int q = 0; q < K; ++q) {
        const uint32_t bw = (q < 8 ? o.b0 : o.b1)[(q >> 1) & 3], cw = (q < 8 ? o.c0 : o.c1)[(q >> 1) & 3];
        const _Float16 bh = __builtin_bit_cast(f16x2, bw)[q & 1], ch = __builtin_bit_cast(f16x2, cw)[q & 1];
        float u = __builtin_fmaf((float)st[q], decay, dequant_h(bh, dtv, mz) * x);
        asm("" : "+v"(u));   // rounded to binary32 here, to binary16 below: never one mixed-precision rounding
        acc[q & 1] = __builtin_fmaf(u, (float)ch, acc[q & 1]);
        st[q] = (_Float16)u;
        if constexpr (STATS) sum[q] = sum[q] + __builtin_fabsf((float)st[q]);
      }
      float y = acc[0] + acc[1];
      y = butterfly_add<0>(y);
      y = butterfly_add<1>(y);
      y = butterfly_add<2>(y);
      if (part == 0) sm.y[i][r] = f2h(y + x * Dh);
    };
    // the operands of the next token are read while this one steps
    Operands o0 = operands(0);
    int i = 0;
    for (; i + 1 < n; i += 2) {
      const Operands o1 = operands(i + 1);
      step(o0, i);
      o0 = operands(min(i + 2, T - 1));
      step(o1, i + 1);
    }
    if (i < n) step(o0, i);
    if (t0 + T < L) stage_block(buf ^ 1);
    __syncthreads();   // the block's readouts are in LDS
    if (xin && xt < n)
      *(u32x4*)(a.y + ((size_t)(b * L + t0 + xt) * H + h) * P + pbase + xp) = *(const u32x4*)&sm.y[xt][xp];
  }
  if (valid) {
    u32x4 v[2];
#pragma unroll
    for (int w = 0; w < 8; ++w)
      v[w >> 2][w & 3] = (uint32_t)__builtin_bit_cast(uint16_t, st[2 * w]) |
                         ((uint32_t)__builtin_bit_cast(uint16_t, st[2 * w + 1]) << 16);
    srow[0] = v[0];
    srow[1] = v[1];
  }
  if constexpr (STATS) {
    // the wave's two 4-row sub-tiles, (r0 + r1) + (r2 + r3) (rows past P add
    // zero), then each 16-row tile as ((T0 + T1) + T2) + T3
#pragma unroll
    for (int i = 0; i < K; ++i) {
      const float s = butterfly_add<4>(add_lane_xor8(valid ? sum[i] : 0.f));
      if ((lane & 24) == 0) sm.sub[wave][lane >> 5][K * part + i] = s;
    }
    __syncthreads();
    const int tl = tid >> 7, nn = tid & 127, tiles = (P + 15) / 16, tile = pbase / 16 + tl;
    if (tile < tiles)
      a.stats[(((size_t)b * H + h) * tiles + tile) * 128 + nn] =
          ((sm.sub[2 * tl][0][nn] + sm.sub[2 * tl][1][nn]) + sm.sub[2 * tl + 1][0][nn]) + sm.sub[2 * tl + 1][1][nn];
  }
}

hipError_t launch_s16_rows(const S16Args& a, hipStream_t stream) {
  const dim3 grid((unsigned)((a.P + S16_ROWS - 1) / S16_ROWS), (unsigned)a.H, (unsigned)a.B);
  if (a.stats) hipLaunchKernelGGL((k_s16_rows<true>), grid, dim3(256), 0, stream, a);
  else hipLaunchKernelGGL((k_s16_rows<false>), grid, dim3(256), 0, stream, a);
  return hipGetLastError();
}

// The scan pays its taking apart and putting together of the rows with the
// first tokens.  us per call, one-lane-per-row kernel / this scan, at batch 1,
// 8 and 64 of 128 heads of 64 rows (128, 1,024 and 8,192 slots):
//   tier 32/32/64     8 tokens 14.4 / 11.3, 20.5 / 20.7, 102.2 / 115.7
//                    16 tokens 24.0 / 14.8, 33.4 / 30.5, 183.1 / 180.5
//   legacy 16/64/48   8 tokens 14.6 / 12.4, 22.2 / 23.0, 136.6 / 150.6
//   tier 8/80/40     16 tokens at batch 8 39.9 / 41.2
//   dense3            2 tokens 11.9 /  9.2,  4: 22.2 / 20.6, 16: 299.9 / 280.2
//   ridge 24/44/60    8 tokens 17.9 / 23.8, 26.2 / 36.9, 145.3 / 146.2
//                    16 tokens 30.8 / 28.2, 46.2 / 48.4, 263.8 / 227.9
//   ridge 8/76/44    24 tokens at batch 4 and 8 52.2 / 50.9, 66.0 / 72.5
// Wide rows over many slots (four lanes per row, see rows_lanes) come out
// even near 64 tokens: tier 8/80/40 at batch 16, 222.0 / 221.0; ridge 8/76/44
// 286 / 273.
// Between 2,048 and 3,072 slots a tier's one lane per row runs in two rounds of
// two waves per SIMD, where the one-lane kernels hold all of them at once:
// 32/32/64 at batch 20, 24 tokens 93.4 / 118.3, 64 tokens 234 / 277, and 24/48/56,
// 36/24/68 and 40/16/72 lose 4 to 27% too, but 44/8/76 wins, 64 tokens 257 / 237.
// At batch 28 32/32/64 takes 124.7 / 129.6 for 24 tokens, 163.4 / 164.3 for 32.
// A head whose rows would leave waves of a workgroup idle (two lanes or one,
// and heads per group that no two or four of them fill it with) stays with the
// one-lane kernels: 8 heads in 8 groups at batch 500, 24 tokens, tier 32/32/64
// 127 / 443.  A ridge scan's records serve the heads of a group: one head per
// group pays from 64 tokens on to 1,280 slots (batch 138: 32 tokens 141 / 144, 64
// 273 / 255), and not above (batch 175, 128 tokens 535 / 566).  Wide rows of two
// or three heads per group gain from 64 tokens on almost everywhere (8/76/44, 16
// heads in 8 groups of 16 rows at batch 345, 105 tokens 1,315 / 913; batch 122 of
// 9 heads in 3, 64 tokens 294 / 214; a loss is batch 333 of 6 in 3, 308 / 343).
int rows_scan_lanes(int mode, int carried, long long B, int L, int H, int P, int G) {
  const long long slots = rows_slots(B, H, P);
  const int lanes = rows_lanes(carried, slots), rows = 64 / lanes, hpg = H / G;
  const int blocks = rows_blocks(lanes, P), heads = rows_heads(blocks, hpg);
  // rows a head takes room for here, and in the one-lane kernels' slots
  const int room = 4 * rows * ((blocks * heads + 3) / 4) / heads;
  if (L < 2 || P % 8 || room > 64 * ((P + 63) / 64)) return 0;
  const bool wide = carried > 72;
  int least;
  if (mode == MODE_DENSE3) {
    least = slots <= 384 ? 2 : slots <= 1024 ? 4 : 16;
  } else if (mode == MODE_RIDGE) {
    if (slots > 1280 && hpg == 1) return 0;
    least = slots > 1024 && hpg == 1 ? 64 : slots <= 256 ? 16 : slots <= 384 ? 20 : slots <= 1024 ? (wide && slots > 768 ? 32 : 24) : wide ? 64 : 24;
  } else {
    if (!wide && carried > 52 && slots > 2048 && slots <= 3072) return 0;
    least = slots <= 384 ? 8 : slots <= 1024 ? (carried > 80 && slots > 768 ? 20 : 16) : wide ? 64
            : slots > 3072 && slots <= 3584 ? 32 : 24;
  }
  return L >= least ? lanes : 0;
}

template <int N8, int N4, int NZ, int MODE>
hipError_t launch_rows(const StepArgs& a, hipStream_t stream) {
  return launch_rows_scan<N8, N4, NZ, MODE>(a, 0, a.L, stream);
}
template hipError_t launch_rows<16, 64, 48, MODE_LEGACY>(const StepArgs&, hipStream_t);
template hipError_t launch_rows<16, 64, 48, MODE_STORED>(const StepArgs&, hipStream_t);
template hipError_t launch_rows<8, 80, 40, MODE_STORED>(const StepArgs&, hipStream_t);
template hipError_t launch_rows<24, 48, 56, MODE_STORED>(const StepArgs&, hipStream_t);
template hipError_t launch_rows<32, 32, 64, MODE_STORED>(const StepArgs&, hipStream_t);
template hipError_t launch_rows<36, 24, 68, MODE_STORED>(const StepArgs&, hipStream_t);
template hipError_t launch_rows<40, 16, 72, MODE_STORED>(const StepArgs&, hipStream_t);
template hipError_t launch_rows<44, 8, 76, MODE_STORED>(const StepArgs&, hipStream_t);

hipError_t launch_dense3_rows(const StepArgs& a, int equalizer, hipStream_t stream) {
  return launch_rows_scan<64, 64, 0, MODE_DENSE3>(a, equalizer, a.L, stream);
}

}  // namespace m2r

using namespace m2r;

extern "C" int m2r_scan_lanes(int codec, int n8, int n4, int64_t batch, int64_t L, int64_t H, int64_t P, int64_t G) {
  if (batch <= 0 || L <= 0 || H <= 0 || P <= 0 || G <= 0 || H % G || n8 < 0 || n4 < 0) return 0;
  if (codec < 0 || codec > 3 || (double)batch * L * H * P >= 2147483647.0) return 0;
  return rows_scan_lanes(codec, codec == MODE_DENSE3 ? 128 : n8 + n4, batch, (int)L, (int)H, (int)P, (int)G);
}
