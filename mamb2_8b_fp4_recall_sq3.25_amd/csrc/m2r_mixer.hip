// One-token causal depthwise convolution update of the Mamba-2 mixer, for
// gfx950: the cached window rolls by one step, takes the new projection
// column, and the output is silu(sum(window * weight) + bias).
//
// Arithmetic: the reference's PyTorch fallback of the update
// (mamba2_recall/state_quant.py:289-297), operation for operation:
//   window <- roll(window, -1) along time; window[..., K-1] <- value
//   p_t = half(window_t * w_t)                 (binary16 products)
//   s   = half(((p_0 + p_1) + p_2) + p_3)      (binary32 sum in time order)
//   s   = half(s + bias)                       (when a bias is given)
//   out = half(s / (1 + exp(-s)))              (silu in binary32)
// One thread per (batch row, channel); the window is read and written
// through its strides (the controller keeps it time-major: [B, K, C] memory).
#include "m2r_device.h"
#include "m2r_abi_util.h"
#include "m2r_tile.h"

#include <initializer_list>

namespace m2r {

template <int K>
__global__ __launch_bounds__(256) void k_conv_update(uint16_t* window, int64_t ws_b, int64_t ws_c, int64_t ws_t,
                                                     const uint16_t* value, int64_t vs_b, const uint16_t* weight,
                                                     const uint16_t* bias, uint16_t* out, int64_t batch,
                                                     int64_t channels, int silu) {
  const int64_t i = (int64_t)blockIdx.x * 256 + threadIdx.x;
  if (i >= batch * channels) return;
  const int64_t b = i / channels, c = i - b * channels;
  uint16_t* w = window + b * ws_b + c * ws_c;
  uint16_t win[K];
#pragma unroll
  for (int t = 0; t < K - 1; ++t) win[t] = w[(t + 1) * ws_t];
  win[K - 1] = value[b * vs_b + c];
  float acc = 0.f;
#pragma unroll
  for (int t = 0; t < K; ++t) {
    w[t * ws_t] = win[t];
    acc = acc + h2f(f2h(h2f(win[t]) * h2f(weight[c * K + t])));
  }
  float s = h2f(f2h(acc));
  if (bias) s = h2f(f2h(s + h2f(bias[c])));
  if (silu) s = s / (1.0f + expf(-s));
  out[i] = f2h(s);
}

}  // namespace m2r

using namespace m2r;

extern "C" int m2r_causal_conv_update(void* window, int64_t ws_b, int64_t ws_c, int64_t ws_t, const void* value,
                                      int64_t vs_b, const void* weight, const void* bias, void* out, int64_t batch,
                                      int64_t channels, int width, int silu, hipStream_t stream) {
  if (batch <= 0 || channels <= 0) return m2r_fail("conv update: non-positive shape");
  if (width != 4) return m2r_fail("conv update: the Mamba-2 convolution width is 4");
  if (batch * channels > (int64_t)1 << 40) return m2r_fail("conv update: size limits");
  const int64_t n = batch * channels;
  hipLaunchKernelGGL(k_conv_update<4>, dim3((unsigned)((n + 255) / 256)), dim3(256), 0, stream, (uint16_t*)window,
                     ws_b, ws_c, ws_t, (const uint16_t*)value, vs_b, (const uint16_t*)weight,
                     (const uint16_t*)bias, (uint16_t*)out, batch, channels, silu);
  return m2r_check(hipGetLastError(), "conv update launch");
}

// ---------------------------------------------------------------------------
// Causal depthwise convolution of several tokens, the prefill form of the
// update above (the PyTorch branch of mamba2_recall/state_quant.py:305-317):
//   s   = half(float(sum_k x[t - 3 + k] * w[k])) (binary64 sum, as the library rounds it)
//   s   = half(s + bias)                       (when a bias is given)
//   out = half(s / (1 + exp(-s)))              (silu in binary32)
// x before the first token is the cached window's last three inputs when the
// request has a history; without one those taps are left out (not multiplied
// by zero).  The window then holds the last four inputs.
//
// Bound: about 45 vector instructions per output (four binary64 products, the
// roundings, exp and divide) next to two bytes read and two written.  As
// library calls this was a transposing copy, a convolution with strided
// stores, a bias pass, a SiLU pass and three copies that split the channels:
// 1024 tokens of 10240 channels took about 160 us of a mixer call, and take
// 18 us here (42 MB, 8 us at the rate of a copy).  A thread keeps the window
// of four neighbouring channels in registers over kConvSeg tokens, reads the
// projection's rows in place and writes x, B and C as the contiguous tensors
// the scan reads.  Eight channels per thread need 167 registers, and 2.5
// waves per SIMD took 22 us.
namespace m2r {

constexpr int kConvSeg = 8;   // tokens per thread: 3 inputs read again per 8, and five waves per SIMD at that size

typedef uint16_t u16x4 __attribute__((ext_vector_type(4)));

struct ConvArgs {
  uint16_t* window;
  int64_t ws_b, ws_t;
  const uint16_t* value;
  int64_t vs_b, vs_l;
  const uint16_t *weight, *bias;
  uint16_t* out[3];
  int64_t n[3];   // channels of each output
  int64_t batch, tokens, segs;
  int history;
};

__global__ __launch_bounds__(256) void k_conv_tokens(ConvArgs a) {
  const int64_t chunks = (a.n[0] + a.n[1] + a.n[2]) / 4;
  int64_t i = (int64_t)blockIdx.x * 256 + threadIdx.x;
  if (i >= chunks * a.segs * a.batch) return;
  const int64_t chunk = i % chunks;
  i /= chunks;
  const int64_t seg = i % a.segs, b = i / a.segs;
  int64_t c = chunk * 4;
  const int64_t t0 = seg * kConvSeg;
  const int64_t left = a.tokens - t0;
  const uint16_t* v = a.value + b * a.vs_b + c;
  double w[4][4];
  {
    const u16x4* wp = (const u16x4*)(a.weight + c * 4);
#pragma unroll
    for (int q = 0; q < 4; ++q) {
      const u16x4 ww = wp[q];
#pragma unroll
      for (int j = 0; j < 4; ++j) w[q][j] = (double)h2f(ww[j]);
    }
  }
  u16x4 bias;
  if (a.bias) bias = *(const u16x4*)(a.bias + c);
  // in[k] is token t0 - 3 + k; `first` of the three before t0 do not exist
  u16x4 in[3 + kConvSeg];
  uint16_t* win = a.window + b * a.ws_b + c;
  int first = 0;
#pragma unroll
  for (int k = 0; k < 3; ++k) in[k] = 0;
  if (seg) {
#pragma unroll
    for (int k = 0; k < 3; ++k) in[k] = *(const u16x4*)(v + (t0 - 3 + k) * a.vs_l);
  } else if (a.history) {
#pragma unroll
    for (int k = 0; k < 3; ++k) in[k] = *(const u16x4*)(win + (k + 1) * a.ws_t);
  } else {
    first = 3;
  }
#pragma unroll
  for (int k = 0; k < kConvSeg; ++k)
    in[3 + k] = *(const u16x4*)(v + (t0 + (k < left ? k : left - 1)) * a.vs_l);
  if (!seg) {
    // the only thread of this batch row and these channels that reads the
    // window also writes it: inputs tokens - 4 .. tokens - 1
#pragma unroll
    for (int k = 0; k < 4; ++k) {
      const int64_t t = a.tokens - 4 + k;
      u16x4 last = t == -3 ? in[0] : t == -2 ? in[1] : in[2];
      if (t >= 0) last = *(const u16x4*)(v + t * a.vs_l);
      *(u16x4*)(win + k * a.ws_t) = last;
    }
  }
  int part = 0;
  if (c >= a.n[0]) { c -= a.n[0]; part = 1; }
  if (part && c >= a.n[1]) { c -= a.n[1]; part = 2; }
  const int64_t pitch = part == 0 ? a.n[0] : part == 1 ? a.n[1] : a.n[2];
  uint16_t* o = (part == 0 ? a.out[0] : part == 1 ? a.out[1] : a.out[2]) + (b * a.tokens + t0) * pitch + c;
#pragma unroll
  for (int k = 0; k < kConvSeg; ++k) {
    if (k >= left) break;
    u16x4 r;
#pragma unroll
    for (int j = 0; j < 4; ++j) {
      double acc = 0.0;
#pragma unroll
      for (int q = 0; q < 4; ++q) {
        const double next = __builtin_fma((double)h2f(in[k + q][j]), w[j][q], acc);
        acc = k + q < 3 && k + q < first ? acc : next;
      }
      float s = h2f(f2h((float)acc));
      if (a.bias) s = h2f(f2h(s + h2f(bias[j])));
      r[j] = f2h(s / (1.0f + expf(-s)));
    }
    *(u16x4*)(o + k * pitch) = r;
  }
}

}  // namespace m2r

extern "C" int m2r_causal_conv_tokens(void* window, int64_t ws_b, int64_t ws_t, int history, const void* value,
                                      int64_t vs_b, int64_t vs_l, const void* weight, const void* bias, void* x,
                                      void* bm, void* cm, int64_t n_x, int64_t n_b, int64_t n_c, int64_t batch,
                                      int64_t tokens, int width, hipStream_t stream) {
  if (batch <= 0 || tokens <= 0 || n_x <= 0 || n_b <= 0 || n_c <= 0) return m2r_fail("conv tokens: non-positive shape");
  if (width != 4) return m2r_fail("conv tokens: the Mamba-2 convolution width is 4");
  const int64_t lim = (int64_t)1 << 30;
  if (batch > lim || tokens > lim || n_x > lim || n_b > lim || n_c > lim)
    return m2r_fail("conv tokens: size limits");
  const int64_t channels = n_x + n_b + n_c, segs = (tokens + kConvSeg - 1) / kConvSeg;
  if ((n_x | n_b | n_c) & 3) return m2r_fail("conv tokens: channel counts must be multiples of 4");
  if (((ws_b | ws_t | vs_b | vs_l) & 3) || ws_t < channels || vs_l < channels)
    return m2r_fail("conv tokens: strides must be multiples of 4 elements, the rows' at least the channel count");
  if (!window || !value || !weight || !x || !bm || !cm) return m2r_fail("conv tokens: null pointer");
  for (const void* p : {(const void*)window, value, weight, bias, (const void*)x, (const void*)bm, (const void*)cm})
    if ((uintptr_t)p & 7) return m2r_fail("conv tokens: operands must be 8-byte aligned");
  const __int128 blocks = ((__int128)(channels / 4) * segs * batch + 255) / 256;
  if (blocks > 0x7fffffff) return m2r_fail("conv tokens: grid limits exceeded");
  ConvArgs a{(uint16_t*)window, ws_b, ws_t, (const uint16_t*)value, vs_b, vs_l, (const uint16_t*)weight,
             (const uint16_t*)bias, {(uint16_t*)x, (uint16_t*)bm, (uint16_t*)cm}, {n_x, n_b, n_c}, batch, tokens,
             segs, history != 0};
  hipLaunchKernelGGL(k_conv_tokens, dim3((unsigned)blocks), dim3(256), 0, stream, a);
  return m2r_check(hipGetLastError(), "conv tokens launch");
}

// ---------------------------------------------------------------------------
// Gated RMS norm of the Mamba-2 mixer (mamba_ssm's RMSNormGated with
// norm_before_gate = False, which the reference's controllers call as
// mx.norm(y, z), mamba2_recall/state_quant.py:298-300), per group of
// `gs` channels of a row, in binary32:
//   v   = y * (z * sigmoid(z)),  sigmoid(z) = 1 / (1 + exp(-z))
//   r   = 1 / sqrt(sum_group(v^2) / gs + eps)
//   out = half((v * r) * weight)
// One 256-thread workgroup per (row, group); a thread holds up to four
// chunks of four channels in registers.  The sum of squares is a fixed tree
// (per thread in chunk order, then the wave's adjacent-pair butterfly, then
// the four waves in order), so results do not vary from run to run.
namespace m2r {

__global__ __launch_bounds__(256) void k_gated_rmsnorm(const uint16_t* y, int64_t ys, const uint16_t* z, int64_t zs,
                                                       const uint16_t* weight, uint16_t* out, int64_t os, int gs,
                                                       float eps) {
  __shared__ float part[4];
  const int64_t row = blockIdx.y;
  const int c0 = blockIdx.x * gs;
  const int tid = threadIdx.x;
  const u16x4* yr = (const u16x4*)(y + row * ys + c0);
  const u16x4* zr = (const u16x4*)(z + row * zs + c0);
  float v[4][4];
  float ss = 0.f;
#pragma unroll
  for (int k = 0; k < 4; ++k) {
    const int q = k * 256 + tid;   // chunk of channels 4q .. 4q + 3 of the group
    if (4 * q < gs) {
      const u16x4 yv = yr[q], zv = zr[q];
#pragma unroll
      for (int j = 0; j < 4; ++j) {
        const float zf = h2f(zv[j]);
        const float sg = 1.0f / (1.0f + expf(-zf));
        v[k][j] = h2f(yv[j]) * (zf * sg);
        ss = __builtin_fmaf(v[k][j], v[k][j], ss);
      }
    }
  }
  ss = wave_sum(ss);
  if ((tid & 63) == 0) part[tid >> 6] = ss;
  __syncthreads();
  const float tot = (part[0] + part[1]) + (part[2] + part[3]);
  const float r = 1.0f / __builtin_sqrtf(tot / (float)gs + eps);
  const u16x4* wr = (const u16x4*)(weight + c0);
  u16x4* orow = (u16x4*)(out + row * os + c0);
#pragma unroll
  for (int k = 0; k < 4; ++k) {
    const int q = k * 256 + tid;
    if (4 * q < gs) {
      const u16x4 wv = wr[q];
      u16x4 o;
#pragma unroll
      for (int j = 0; j < 4; ++j) o[j] = f2h((v[k][j] * r) * h2f(wv[j]));
      orow[q] = o;
    }
  }
}

}  // namespace m2r

extern "C" int m2r_gated_rmsnorm(const void* y, int64_t y_stride, const void* z, int64_t z_stride,
                                 const void* weight, void* out, int64_t out_stride, int64_t rows, int64_t channels,
                                 int64_t group_size, float eps, hipStream_t stream) {
  if (rows <= 0 || channels <= 0 || group_size <= 0) return m2r_fail("gated norm: non-positive shape");
  if (channels % group_size) return m2r_fail("gated norm: channels must be a multiple of the group size");
  if (group_size % 4 || group_size > 4096) return m2r_fail("gated norm: group size must be a multiple of 4, at most 4096");
  if (rows > 65535 || channels / group_size > 65535) return m2r_fail("gated norm: grid limits exceeded");
  if (!(eps >= 0.f)) return m2r_fail("gated norm: eps must be non-negative");
  if (!y || !z || !weight || !out) return m2r_fail("gated norm: null pointer");
  for (const void* p : {y, z, weight, (const void*)out})
    if ((uintptr_t)p & 7) return m2r_fail("gated norm: y, z, weight and out must be 8-byte aligned");
  if ((y_stride | z_stride | out_stride) & 3 || y_stride < channels || z_stride < channels || out_stride < channels)
    return m2r_fail("gated norm: row strides must be multiples of 4 elements, at least the channel count");
  hipLaunchKernelGGL(k_gated_rmsnorm, dim3((unsigned)(channels / group_size), (unsigned)rows), dim3(256), 0, stream,
                     (const uint16_t*)y, y_stride, (const uint16_t*)z, z_stride, (const uint16_t*)weight,
                     (uint16_t*)out, out_stride, (int)group_size, eps);
  return m2r_check(hipGetLastError(), "gated norm launch");
}
