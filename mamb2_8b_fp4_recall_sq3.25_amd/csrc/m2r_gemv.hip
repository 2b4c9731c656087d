// Packed-resident FP4 (E2M1, G16) matrix-vector products for gfx950:
// y[m, n] = sum_k u[m, k] * w[n, k] for M <= 4 activation rows, with the
// weights read straight from the checkpoint format (two codes per byte, one
// E4M3 block scale per 16 weights, one FP32 global scale) instead of from a
// decoded FP16 copy: 0.5625 bytes per weight instead of 2.
//
// Every weight is the binary16 value fp4.decode_packet produces
// (mamba2_recall/fp4.py:151-154): half(RN(RN(lev * block) * global)), lev in
// {0, .5, 1, 1.5, 2, 3, 4, 6}, sign from bit 3 of the code.  Each workgroup
// builds that value for every (block byte, level) pair in an LDS table (128 x
// 8 binary16, stored as low-byte and high-byte planes), so a weight costs one
// byte-permute lookup: the code nibbles select their entries' low and high
// bytes with v_perm_b32, each code's sign bit is or-ed into bit 7 of its high
// byte (the binary16 sign), two more permutes form the binary16 pairs, and
// v_dot2_f32_f16 multiplies weight pairs by activation pairs and accumulates
// in binary32: about 2.25 VALU instructions per weight and activation row.  The packet must satisfy decode_packet's checks
// (the loader validates each matrix once); block bytes with the sign bit set
// other than 0x80 are outside that contract.
//
// Mapping: a workgroup of four waves takes 4 / KCH rows at a time (rows
// strided over the grid); wave w works on 2048-wide chunk c = w % KCH of row
// w / KCH, lane l on k in [2048 c + 32 l, 2048 c + 32 l + 32): one 16-byte
// code load, one 2-byte scale load and two table reads per row.  The loads of
// the next two rows are in flight while a row computes; the grid is one
// resident round of workgroups.  The activations of the
// lane's k range stay in registers, reordered once into the weight pairs'
// order.  A wave sum per chunk, then the chunks' partial sums in a fixed
// order through LDS, finish each output.  One activation row (the batch-1
// decode) takes k_fp4_gemv_rows instead where it fills the chip in one
// resident round: whole rows per wave, no barrier per row, the same sums.  Four
// rows take k_fp4_gemv_tiles (matrix cores) where their outputs fill enough of
// the chip; it sums in another order, so a row's bits are those of one or two
// rows only below that.
#include "m2r_device.h"
#include "m2r_abi_util.h"
#include "m2r_tile.h"

#include <algorithm>
#include <atomic>

namespace m2r {

typedef _Float16 gh2 __attribute__((ext_vector_type(2)));

__device__ __forceinline__ float dot2(uint32_t a, uint32_t b, float c) {
  return __builtin_amdgcn_fdot2(__builtin_bit_cast(gh2, a), __builtin_bit_cast(gh2, b), c, false);
}

// 8 weights of code word cw against the activation pairs ue (k = 0,2 | 4,6)
// and uo (1,3 | 5,7) of the same 8 positions, with the block's table t.
__device__ __forceinline__ void fp4_dot8(uint32_t cw, const uint32_t (&t)[4], const uint32_t* ue, const uint32_t* uo,
                                         float& acc) {
  const uint32_t even = cw & 0x07070707u, odd = (cw >> 4) & 0x07070707u;
  // low and high bytes of the magnitudes; the code's sign bit (bit 3 of the
  // nibble: bit 3 of byte j for the even weight 2j, bit 7 for the odd weight
  // 2j+1) becomes bit 7 of the high byte, i.e. the binary16 sign (the
  // magnitudes' high bytes have it clear)
  const uint32_t le = __builtin_amdgcn_perm(t[1], t[0], even), lo = __builtin_amdgcn_perm(t[1], t[0], odd);
  const uint32_t he = __builtin_amdgcn_perm(t[3], t[2], even) | ((cw & 0x08080808u) << 4);
  const uint32_t ho = __builtin_amdgcn_perm(t[3], t[2], odd) | (cw & 0x80808080u);
  // binary16 pairs (w0, w2), (w4, w6), (w1, w3), (w5, w7): low byte, high byte
  const uint32_t e01 = __builtin_amdgcn_perm(he, le, 0x05010400u), e23 = __builtin_amdgcn_perm(he, le, 0x07030602u);
  const uint32_t o01 = __builtin_amdgcn_perm(ho, lo, 0x05010400u), o23 = __builtin_amdgcn_perm(ho, lo, 0x07030602u);
  acc = dot2(e01, ue[0], acc);
  acc = dot2(e23, ue[1], acc);
  acc = dot2(o01, uo[0], acc);
  acc = dot2(o23, uo[1], acc);
}

template <int M, int KCH>
__global__ __launch_bounds__(256) void k_fp4_gemv(const uint8_t* __restrict__ codes, const uint8_t* __restrict__ scales,
                                                  const float* __restrict__ gscale, const uint16_t* __restrict__ u,
                                                  int64_t u_stride, uint16_t* __restrict__ y, int64_t y_stride,
                                                  int N) {
  static_assert(KCH == 1 || KCH == 2 || KCH == 4, "the four waves split a row's chunks evenly");
  constexpr int K = KCH * 2048;
  constexpr int RPI = 4 / KCH;   // rows per workgroup iteration: wave w takes chunk w % KCH of row w / KCH
  __shared__ __align__(16) uint32_t s_tab[128][4];   // per block byte: low bytes of T[0..7], then high bytes
  __shared__ float s_part[2][RPI][KCH][M];           // per-chunk partial sums, double-buffered by iteration
  const int lane = threadIdx.x & 63;
  const int wave = threadIdx.x >> 6;
  const int c = wave % KCH, r = wave / KCH;
  const int stride = (int)gridDim.x * RPI;
  int n = (int)blockIdx.x * RPI + r;
  // the first row's loads go out before the table is built
  auto load_row = [&](int row, u32x4& cv, uint32_t& sb) {
    const int rr = min(row, N - 1);   // rows past N re-read row N-1 (never stored)
    cv = __builtin_nontemporal_load((const u32x4*)(codes + (size_t)rr * (K / 2) + c * 1024) + lane);
    sb = *(const uint16_t*)(scales + (size_t)rr * (K / 16) + c * 128 + 2 * lane);
  };
  // two rows ahead: the loads of iterations it + 1 and it + 2 are in flight
  // while iteration it computes
  u32x4 cv, cv2;
  uint32_t sb, sb2;
  load_row(n, cv, sb);
  load_row(n + stride, cv2, sb2);
  const float gl = *gscale;
  for (int e = threadIdx.x; e < 128 * 8; e += 256) {
    const int blk = e >> 3, i = e & 7;
    // 2 * lev as an integer, times block / 2: RN(lev * block) exactly
    const float lev2 = (float)((i < 4) ? i : (i == 4 ? 4 : (i == 5 ? 6 : (i == 6 ? 8 : 12))));
    const float hb = e4m3_byte_to_f32<0>((uint32_t)blk) * 0.5f;
    const uint16_t h = f2h((lev2 * hb) * gl);
    uint8_t* row = (uint8_t*)s_tab[blk];
    row[i] = (uint8_t)(h & 0xFFu);
    row[8 + i] = (uint8_t)(h >> 8);
  }
  // activations of the lane's k range of chunk c, as pairs in the weights'
  // order: per 8 positions (u0,u2), (u4,u6) | (u1,u3), (u5,u7)
  uint32_t ue[M][8], uo[M][8];
#pragma unroll
  for (int m = 0; m < M; ++m) {
    const uint32_t* src = (const uint32_t*)(u + m * u_stride + c * 2048 + 32 * lane);
    uint32_t p[16];
#pragma unroll
    for (int q = 0; q < 4; ++q) {
      const u32x4 v = ((const u32x4*)src)[q];
      p[4 * q] = v.x; p[4 * q + 1] = v.y; p[4 * q + 2] = v.z; p[4 * q + 3] = v.w;
    }
#pragma unroll
    for (int q = 0; q < 4; ++q) {   // 8 positions = natural pairs p[4q .. 4q+3]
      ue[m][2 * q] = __builtin_amdgcn_perm(p[4 * q + 1], p[4 * q], 0x05040100u);
      ue[m][2 * q + 1] = __builtin_amdgcn_perm(p[4 * q + 3], p[4 * q + 2], 0x05040100u);
      uo[m][2 * q] = __builtin_amdgcn_perm(p[4 * q + 1], p[4 * q], 0x07060302u);
      uo[m][2 * q + 1] = __builtin_amdgcn_perm(p[4 * q + 3], p[4 * q + 2], 0x07060302u);
    }
  }
  __syncthreads();   // the table is complete
  for (int it = 0; (int)blockIdx.x * RPI + it * stride < N; ++it) {
    const u32x4 cur = cv;
    const uint32_t scur = sb;
    cv = cv2;
    sb = sb2;
    load_row(n + 2 * stride, cv2, sb2);
    float acc[M];
#pragma unroll
    for (int m = 0; m < M; ++m) acc[m] = 0.f;
#pragma unroll
    for (int gidx = 0; gidx < 2; ++gidx) {   // two 16-weight groups per lane
      const u32x4 tv = *(const u32x4*)s_tab[(scur >> (8 * gidx)) & 0x7Fu];
      const uint32_t t[4] = {tv.x, tv.y, tv.z, tv.w};
#pragma unroll
      for (int h = 0; h < 2; ++h) {
        const int q = 2 * gidx + h;   // code word of the 16-byte load: positions 8q .. 8q+7
        const uint32_t cw = q == 0 ? cur.x : q == 1 ? cur.y : q == 2 ? cur.z : cur.w;
#pragma unroll
        for (int m = 0; m < M; ++m) fp4_dot8(cw, t, &ue[m][2 * q], &uo[m][2 * q], acc[m]);
      }
    }
    float (&part)[RPI][KCH][M] = s_part[it & 1];
#pragma unroll
    for (int m = 0; m < M; ++m) {
      const float sum = wave_sum(acc[m]);
      if (lane == 0) part[r][c][m] = sum;
    }
    __syncthreads();   // one barrier per iteration: the other buffer is free again by the next one
    if (c == 0 && lane < M && n < N) {
      float tot = part[r][0][lane];
#pragma unroll
      for (int cc = 1; cc < KCH; ++cc) tot += part[r][cc][lane];
      y[lane * y_stride + n] = f2h(tot);
    }
    n += stride;
  }
}

// One activation row (M == 1): each wave takes D whole rows (rows strided
// over every wave of the grid, W waves: rows w, w + W, ..., w + (D - 1) W),
// lane l the same k ranges as above in each of the row's KCH chunks, so a row
// needs no workgroup barrier: the KCH chunk sums are wave sums added in chunk
// order, the same bits as k_fp4_gemv<1, KCH>.  The host sizes the grid so
// that D W >= N with every workgroup resident at once: all of a wave's loads
// are issued first (rows past N re-read row N - 1, which is never stored),
// then the table is built, and each row is computed as soon as its loads
// have landed, while the later rows' loads are still in flight.
template <int KCH, int D, int WPB>
__global__ __launch_bounds__(64 * WPB) void k_fp4_gemv_rows(const uint8_t* __restrict__ codes,
                                                           const uint8_t* __restrict__ scales,
                                                           const float* __restrict__ gscale,
                                                           const uint16_t* __restrict__ u,
                                                           uint16_t* __restrict__ y, int N) {
  static_assert(KCH == 1 || KCH == 2 || KCH == 4, "K of 2048, 4096 or 8192");
  constexpr int K = KCH * 2048;
  __shared__ __align__(16) uint32_t s_tab[128][4];
  const int lane = threadIdx.x & 63;
  const int wave = threadIdx.x >> 6;
  const int W = (int)gridDim.x * WPB;
  const int n0 = (int)blockIdx.x * WPB + wave;
  // the activations first (shared by every wave, cache hits), so that
  // waiting for them does not wait for the rows
  u32x4 uv[KCH][4];
#pragma unroll
  for (int cc = 0; cc < KCH; ++cc)
#pragma unroll
    for (int q = 0; q < 4; ++q) uv[cc][q] = ((const u32x4*)(u + cc * 2048 + 32 * lane))[q];
  u32x4 cv[D][KCH];
  uint32_t sb[D][KCH];
#pragma unroll
  for (int j = 0; j < D; ++j) {
    const int row = min(n0 + j * W, N - 1);
#pragma unroll
    for (int cc = 0; cc < KCH; ++cc) {
      cv[j][cc] = __builtin_nontemporal_load((const u32x4*)(codes + (size_t)row * (K / 2) + cc * 1024) + lane);
      sb[j][cc] = *(const uint16_t*)(scales + (size_t)row * (K / 16) + cc * 128 + 2 * lane);
    }
  }
  const float gl = *gscale;
  for (int e = threadIdx.x; e < 128 * 8; e += 64 * WPB) {
    const int blk = e >> 3, i = e & 7;
    const float lev2 = (float)((i < 4) ? i : (i == 4 ? 4 : (i == 5 ? 6 : (i == 6 ? 8 : 12))));
    const float hb = e4m3_byte_to_f32<0>((uint32_t)blk) * 0.5f;
    const uint16_t h = f2h((lev2 * hb) * gl);
    uint8_t* row = (uint8_t*)s_tab[blk];
    row[i] = (uint8_t)(h & 0xFFu);
    row[8 + i] = (uint8_t)(h >> 8);
  }
  // activation pairs in the weights' order: per 8 positions (u0,u2), (u4,u6)
  // | (u1,u3), (u5,u7)
  uint32_t ue[KCH][8], uo[KCH][8];
#pragma unroll
  for (int cc = 0; cc < KCH; ++cc) {
    uint32_t p[16];
#pragma unroll
    for (int q = 0; q < 4; ++q) {
      p[4 * q] = uv[cc][q].x; p[4 * q + 1] = uv[cc][q].y; p[4 * q + 2] = uv[cc][q].z; p[4 * q + 3] = uv[cc][q].w;
    }
#pragma unroll
    for (int q = 0; q < 4; ++q) {
      ue[cc][2 * q] = __builtin_amdgcn_perm(p[4 * q + 1], p[4 * q], 0x05040100u);
      ue[cc][2 * q + 1] = __builtin_amdgcn_perm(p[4 * q + 3], p[4 * q + 2], 0x05040100u);
      uo[cc][2 * q] = __builtin_amdgcn_perm(p[4 * q + 1], p[4 * q], 0x07060302u);
      uo[cc][2 * q + 1] = __builtin_amdgcn_perm(p[4 * q + 3], p[4 * q + 2], 0x07060302u);
    }
  }
  __syncthreads();   // the table is complete
#pragma unroll
  for (int j = 0; j < D; ++j) {
    float tot = 0.f;
#pragma unroll
    for (int cc = 0; cc < KCH; ++cc) {
      const u32x4 cur = cv[j][cc];
      const uint32_t scur = sb[j][cc];
      float acc = 0.f;
#pragma unroll
      for (int gidx = 0; gidx < 2; ++gidx) {
        const u32x4 tv = *(const u32x4*)s_tab[(scur >> (8 * gidx)) & 0x7Fu];
        const uint32_t t[4] = {tv.x, tv.y, tv.z, tv.w};
#pragma unroll
        for (int h = 0; h < 2; ++h) {
          const int q = 2 * gidx + h;
          const uint32_t cw = q == 0 ? cur.x : q == 1 ? cur.y : q == 2 ? cur.z : cur.w;
          fp4_dot8(cw, t, &ue[cc][2 * q], &uo[cc][2 * q], acc);
        }
      }
      const float sum = wave_sum(acc);
      tot = cc == 0 ? sum : tot + sum;
    }
    const int n = n0 + j * W;
    if (lane == 0 && n < N) y[n] = f2h(tot);
  }
}

// Four activation rows: with a dot product per row and weight pair the vector
// units have 3.75 instructions a weight, 1.75 of which form it, and the sums of
// four rows; the matrix cores take the products and sums off them.  A
// workgroup of NW waves takes tiles of 16 matrix rows, wave w the w-th part of
// K, as v_mfma_f32_16x16x32_f16 with the 16 rows of weights (A) against the
// four activation rows (B; the other 12 columns repeat the last one, unused).
// A lane's eight k of an A operand are one code word, in the order in which
// the permutes leave them; the B fragments stay in registers for every tile,
// reordered once to match.  One workgroup per CU, AHEAD tiles of loads in
// flight; the waves' partial sums of up to eight tiles wait in LDS for one
// barrier.  us per launch, dot products / tiles: [18560, 4096] 23.7 / 15.8,
// [4096, 8192] 16.7 / 11.4, [18560, 2048] 16.9 / 8.7, [4096, 4096] 12.9 / 6.5,
// [64000, 4096] 61.1 / 39.5.  (One and two rows keep the dot products: one
// row 14.1 / 15.7 and 8.2 / 10.9 on the first two, and two sum as one does.)
// More tiles ahead or waves per workgroup, and conflict-free table reads,
// measure the same: what bounds it is issuing the 14 vector instructions per
// code word, with the matrix instructions between them.
constexpr int GEMV_TILES = 8;   // tiles whose partial sums wait in LDS for one barrier
typedef _Float16 gh8 __attribute__((ext_vector_type(8)));

template <int KCH, int NW, int AHEAD>
__global__ __launch_bounds__(64 * NW) __attribute__((amdgpu_waves_per_eu(NW == 16 ? 4 : 2, 8)))
void k_fp4_gemv_tiles(const uint8_t* __restrict__ codes, const uint8_t* __restrict__ scales,
                      const float* __restrict__ gscale, const uint16_t* __restrict__ u, int64_t u_stride,
                      uint16_t* __restrict__ y, int64_t y_stride, int N) {
  constexpr int M = 4;
  constexpr int K = KCH * 2048, KW = K / NW, I = KW / 128;
  __shared__ __align__(16) uint32_t s_tab[128][4];
  __shared__ __align__(16) float s_part[GEMV_TILES][NW][16][4];
  const int lane = threadIdx.x & 63, wave = threadIdx.x >> 6;
  const int c16 = lane & 15, g = lane >> 4;
  const int k0 = wave * KW + 32 * g;   // the lane's first k; its pieces of 32 lie 128 apart
  const int tiles = (N + 15) / 16, stride = gridDim.x;
  u32x4 cv[AHEAD][I];
  uint32_t sb[AHEAD][I];
  auto load_tile = [&](int tile, u32x4 (&c)[I], uint32_t (&s)[I]) {
    const int row = min(16 * tile + c16, N - 1);   // rows past N re-read row N-1 (never stored)
    const uint8_t* pc = codes + (size_t)row * (K / 2) + k0 / 2;
    const uint8_t* ps = scales + (size_t)row * (K / 16) + k0 / 16;
#pragma unroll
    for (int i = 0; i < I; ++i) {
      c[i] = *(const u32x4*)(pc + 64 * i);
      s[i] = *(const uint16_t*)(ps + 8 * i);
    }
  };
  // the activations first (cache hits, shared by every workgroup), so that
  // waiting for them does not wait for the tiles.  Columns past M repeat the
  // last row (their products are never stored).
  u32x4 uv[I][4];
  const uint16_t* pu = u + min(c16, M - 1) * u_stride + k0;
#pragma unroll
  for (int i = 0; i < I; ++i)
#pragma unroll
    for (int j = 0; j < 4; ++j) uv[i][j] = *(const u32x4*)(pu + 128 * i + 8 * j);
#pragma unroll
  for (int p = 0; p < AHEAD; ++p)
    if ((int)blockIdx.x + p * stride < tiles) load_tile(blockIdx.x + p * stride, cv[p], sb[p]);
  const float gl = *gscale;
  for (int e = threadIdx.x; e < 128 * 8; e += 64 * NW) {
    const int blk = e >> 3, i = e & 7;
    const float lev2 = (float)((i < 4) ? i : (i == 4 ? 4 : (i == 5 ? 6 : (i == 6 ? 8 : 12))));
    const float hb = e4m3_byte_to_f32<0>((uint32_t)blk) * 0.5f;
    const uint16_t h = f2h((lev2 * hb) * gl);
    uint8_t* row = (uint8_t*)s_tab[blk];
    row[i] = (uint8_t)(h & 0xFFu);
    row[8 + i] = (uint8_t)(h >> 8);
  }
  // pairs in the weights' order: (u0,u2), (u4,u6), (u1,u3), (u5,u7)
  gh8 bf[I][4];
#pragma unroll
  for (int i = 0; i < I; ++i)
#pragma unroll
    for (int j = 0; j < 4; ++j) {
      const u32x4 v = uv[i][j];
      const u32x4 r = {__builtin_amdgcn_perm(v.y, v.x, 0x05040100u), __builtin_amdgcn_perm(v.w, v.z, 0x05040100u),
                       __builtin_amdgcn_perm(v.y, v.x, 0x07060302u), __builtin_amdgcn_perm(v.w, v.z, 0x07060302u)};
      bf[i][j] = __builtin_bit_cast(gh8, r);
    }
  __syncthreads();   // the table is complete
  for (int first = blockIdx.x; first < tiles; first += GEMV_TILES * stride) {
    for (int t0 = 0; t0 < GEMV_TILES && first + t0 * stride < tiles; t0 += AHEAD) {
#pragma unroll
      for (int p = 0; p < AHEAD; ++p) {
        const int t = t0 + p, tile = first + t * stride;
        if (tile < tiles) {
          f32x4 acc[2] = {{0.f, 0.f, 0.f, 0.f}, {0.f, 0.f, 0.f, 0.f}};
#pragma unroll
          for (int i = 0; i < I; ++i)
#pragma unroll
            for (int j = 0; j < 4; ++j) {
              const u32x4 tv = *(const u32x4*)s_tab[(sb[p][i] >> (8 * (j >> 1))) & 0x7Fu];
              const uint32_t cw = cv[p][i][j];
              const uint32_t even = cw & 0x07070707u, odd = (cw >> 4) & 0x07070707u;
              const uint32_t le = __builtin_amdgcn_perm(tv.y, tv.x, even), lo = __builtin_amdgcn_perm(tv.y, tv.x, odd);
              const uint32_t he = __builtin_amdgcn_perm(tv.w, tv.z, even) | ((cw & 0x08080808u) << 4);
              const uint32_t ho = __builtin_amdgcn_perm(tv.w, tv.z, odd) | (cw & 0x80808080u);
              const u32x4 w = {__builtin_amdgcn_perm(he, le, 0x05010400u), __builtin_amdgcn_perm(he, le, 0x07030602u),
                               __builtin_amdgcn_perm(ho, lo, 0x05010400u), __builtin_amdgcn_perm(ho, lo, 0x07030602u)};
              acc[j & 1] =
                  __builtin_amdgcn_mfma_f32_16x16x32_f16(__builtin_bit_cast(gh8, w), bf[i][j], acc[j & 1], 0, 0, 0);
            }
          if (tile + AHEAD * stride < tiles) load_tile(tile + AHEAD * stride, cv[p], sb[p]);
          const f32x4 sum = acc[0] + acc[1];   // rows 4 g .. 4 g + 3 of column c16
          if (c16 < 4) {
#pragma unroll
            for (int q = 0; q < 4; ++q) s_part[t][wave][4 * g + q][c16] = sum[q];
          }
        }
      }
    }
    __syncthreads();
    // output (tile t, row m of y, weight row): the waves' sums in order
    for (int e = threadIdx.x; e < GEMV_TILES * 64; e += 64 * NW) {
      const int t = e >> 6, m = (e >> 4) & 3, row = e & 15, n = 16 * (first + t * stride) + row;
      if (m < M && n < N) {
        float s = s_part[t][0][row][m];
#pragma unroll
        for (int w = 1; w < NW; ++w) s = s + s_part[t][w][row][m];
        y[m * y_stride + n] = f2h(s);
      }
    }
    __syncthreads();
  }
}

}  // namespace m2r

using namespace m2r;

// The whole-row kernel for one activation row: the smallest rows-per-wave D
// for which one resident round of eight-wave workgroups covers N rows, if
// that round has a workgroup for every CU (D <= 6; D <= 2 for K = 8192,
// whose larger D leave two waves per SIMD, slower than the general kernel).
// Returns 1 when launched, 0 when the general kernel is to be used, or a
// negative error.
template <int KCH, int D>
static int launch_rows_d(const uint8_t* packed, const uint8_t* sc, const float* gs, const uint16_t* u, uint16_t* y,
                         int64_t N, int cus, hipStream_t stream) {
  constexpr int WPB = 8;
  // resident workgroups per CU of this instance (a property of the code
  // object, the same on every gfx950 device), queried once
  static std::atomic<int> per_cu_cache{-1};
  int per_cu = per_cu_cache.load(std::memory_order_relaxed);
  if (per_cu < 0) {
    int b = 0;
    if (hipOccupancyMaxActiveBlocksPerMultiprocessor(&b, (const void*)k_fp4_gemv_rows<KCH, D, WPB>, 64 * WPB, 0) !=
        hipSuccess)
      return -m2r_fail("fp4 gemv: occupancy query failed");
    per_cu = b;
    per_cu_cache.store(b, std::memory_order_relaxed);
  }
  const int64_t waves = (N + D - 1) / D, blocks = (waves + WPB - 1) / WPB;
  if (per_cu <= 0 || blocks > (int64_t)per_cu * cus || blocks < cus) return 0;
  hipLaunchKernelGGL((k_fp4_gemv_rows<KCH, D, WPB>), dim3((unsigned)blocks), dim3(64 * WPB), 0, stream, packed, sc,
                     gs, u, y, (int)N);
  return 1;
}

template <int KCH>
static int launch_rows_k(const uint8_t* packed, const uint8_t* sc, const float* gs, const uint16_t* u, uint16_t* y,
                         int64_t N, int cus, hipStream_t stream) {
  int r = 0;
  if (!r) r = launch_rows_d<KCH, 1>(packed, sc, gs, u, y, N, cus, stream);
  if (!r) r = launch_rows_d<KCH, 2>(packed, sc, gs, u, y, N, cus, stream);
  if constexpr (KCH < 4) {
    if (!r) r = launch_rows_d<KCH, 3>(packed, sc, gs, u, y, N, cus, stream);
    if (!r) r = launch_rows_d<KCH, 4>(packed, sc, gs, u, y, N, cus, stream);
    if (!r) r = launch_rows_d<KCH, 5>(packed, sc, gs, u, y, N, cus, stream);
    if (!r) r = launch_rows_d<KCH, 6>(packed, sc, gs, u, y, N, cus, stream);
  }
  return r;
}

static int launch_rows(int kch, const uint8_t* packed, const uint8_t* sc, const float* gs, const uint16_t* u,
                       uint16_t* y, int64_t N, hipStream_t stream) {
  int dev = 0, cus = 0;
  if (hipGetDevice(&dev) != hipSuccess ||
      hipDeviceGetAttribute(&cus, hipDeviceAttributeMultiprocessorCount, dev) != hipSuccess || cus <= 0)
    return -m2r_fail("fp4 gemv: device query failed");
  if (kch == 1) return launch_rows_k<1>(packed, sc, gs, u, y, N, cus, stream);
  if (kch == 2) return launch_rows_k<2>(packed, sc, gs, u, y, N, cus, stream);
  return launch_rows_k<4>(packed, sc, gs, u, y, N, cus, stream);
}

extern "C" int m2r_fp4_gemv_g16(const uint8_t* packed, const uint8_t* e4m3_scales, const float* global_scale,
                                const void* u, int64_t u_stride, void* y, int64_t y_stride, int64_t M, int64_t N,
                                int64_t K, hipStream_t stream) {
  if (M <= 0 || N <= 0 || K <= 0) return m2r_fail("fp4 gemv: non-positive shape");
  if (K % 2048) return m2r_fail("fp4 gemv: K must be a multiple of 2048");
  if (N > (1 << 30) || u_stride < K || y_stride < N) return m2r_fail("fp4 gemv: size or stride limits");
  if ((((uintptr_t)packed | (uintptr_t)u) & 15) || (u_stride % 8) || ((uintptr_t)e4m3_scales & 1))
    return m2r_fail("fp4 gemv: codes and activation rows must be 16-byte aligned, scales 2-byte aligned");
  const int kch = (int)(K / 2048);
  int cus = 0;
  if (M == 4) {
    int dev = 0;
    if (hipGetDevice(&dev) != hipSuccess ||
        hipDeviceGetAttribute(&cus, hipDeviceAttributeMultiprocessorCount, dev) != hipSuccess || cus <= 0)
      return m2r_fail("fp4 gemv: device query failed");
  }
  // Four rows: the matrix cores where half the CUs have a tile of 16 outputs.
  // A workgroup loads all of the activations before its first tile and takes a
  // whole tile's K, so with fewer tiles the dot products, which spread the
  // outputs over every CU, are faster: us per launch, dot products / tiles, for
  // 1,024, 1,536 and 2,048 outputs: K = 4096 4.9 / 5.9, 5.9 / 6.0, 6.8 / 6.0, K =
  // 8192 7.0 / 10.1, 9.5 / 10.1, 11.7 / 10.1.  With K = 2048 the tiles are never
  // slower (64 outputs 3.8 / 3.8, 1,536 4.9 / 4.0).
  const int64_t tiles = (N + 15) / 16;
  if (M == 4 && (kch == 1 || 2 * tiles >= cus)) {
    const dim3 grid((unsigned)std::min<int64_t>(tiles, cus));
#define M2R_TILES(KK, NW, AHEAD)                                                                              \
    if (kch == KK) {                                                                                          \
      hipLaunchKernelGGL((k_fp4_gemv_tiles<KK, NW, AHEAD>), grid, dim3(64 * NW), 0, stream, packed,           \
                         e4m3_scales, global_scale, (const uint16_t*)u, u_stride, (uint16_t*)y, y_stride,     \
                         (int)N);                                                                             \
      return m2r_check(hipGetLastError(), "fp4 gemv launch");                                                 \
    }
    M2R_TILES(1, 8, 2) M2R_TILES(2, 8, 2) M2R_TILES(4, 16, 1)
#undef M2R_TILES
  }
  if (M == 1) {
    if (int e = launch_rows(kch, packed, e4m3_scales, global_scale, (const uint16_t*)u, (uint16_t*)y, N, stream))
      return e > 0 ? m2r_check(hipGetLastError(), "fp4 gemv launch") : 1;
  }
  const int rpi = 4 / kch > 0 ? 4 / kch : 1;
  // one resident round: eight four-wave workgroups per CU
  const int blocks = (int)std::min<int64_t>((N + rpi - 1) / rpi, 2048);
  const dim3 grid(blocks), block(256);
#define M2R_GEMV(MM, KK)                                                                                       \
  if (M == MM && kch == KK) {                                                                                  \
    hipLaunchKernelGGL((k_fp4_gemv<MM, KK>), grid, block, 0, stream, packed, e4m3_scales, global_scale,         \
                       (const uint16_t*)u, u_stride, (uint16_t*)y, y_stride, (int)N);                          \
    return m2r_check(hipGetLastError(), "fp4 gemv launch");                                                   \
  }
  M2R_GEMV(1, 1) M2R_GEMV(1, 2) M2R_GEMV(1, 4)
  M2R_GEMV(2, 1) M2R_GEMV(2, 2) M2R_GEMV(2, 4)
  M2R_GEMV(4, 2) M2R_GEMV(4, 4)
#undef M2R_GEMV
  return m2r_fail("fp4 gemv: supported are M in {1, 2, 4} rows of u and K in {2048, 4096, 8192}");
}
