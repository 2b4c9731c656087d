// Multi-token scans with each state row spread over several lanes
// (m2r_rows.hip): arguments and launchers, called by the codecs' entry points.
#pragma once
#include <hip/hip_runtime.h>
#include <stdint.h>

namespace m2r {

struct S16Args {
  const uint16_t* x; const uint16_t* dt; const float* A; const uint16_t* Bm; const uint16_t* Cm;
  const void* D; const void* dt_bias;
  uint16_t* state; uint16_t* y; float* stats;
  int B, L, H, P, G;
  int d_f32, db_f32;
};

// The scan of an FP16 carry over a.L > 1 tokens, with statistics where
// a.stats is not null.  P % 8 == 0; x, B, C, state and y 16-byte aligned.
hipError_t launch_s16_rows(const S16Args& a, hipStream_t stream);

// The scan of packed rows over a.L > 1 tokens (m2r_rows_kernel.h); a ridge
// scan first writes its token records to a.rec.  StepArgs::dma_tiles bit 0
// set; x, B, C and y 16-byte aligned.  Defined for the layouts of the packed
// codecs in m2r_rows.hip and m2r_rows_ridge.hip.
struct StepArgs;

// 64-row slots of a scan.
inline long long rows_slots(long long B, int H, int P) { return B * H * ((P + 63) / 64); }

// Lanes per row, by the scan's 64-row slots: enough to give every SIMD a
// wave, then fewer, as each lane repeats a token's scalar work.  us for 64
// tokens at batch 1, 3, 4, 8, 12, 16 and 64 (128 slots each), ridge 24/44/60:
//   8 lanes   56.3   84.0  105.6  172.5  244.4  316.9
//   4         78.7   90.6   91.7  155.2  198.0  255.0    923
//   2        105.8  108.8  109.7  128.9  210.2  236.0    880
//   1        162.2  164.2  164.0  174.5  196.3  203.4    753
// One lane has all carried coordinates and updates in registers: with more
// than 72 they spill (8/76/44 at batch 16: 279 against 273 on four lanes).
inline int rows_lanes(int carried, long long slots) {
  if (slots <= 384) return 8;
  if (slots <= 768) return 4;
  if (slots <= 1024) return 2;
  return slots <= 1536 || carried > 72 ? 4 : 1;
}

// A workgroup's four waves take blocks of 64 / lanes rows of one head where it
// has enough of them, else of two or four heads of one group.
inline int rows_blocks(int lanes, int P) { return (P + 64 / lanes - 1) / (64 / lanes); }
inline int rows_heads(int blocks, int hpg) {
  return blocks == 1 && hpg % 4 == 0 ? 4 : blocks <= 2 && hpg % 2 == 0 ? 2 : 1;
}

// Lanes per row of the row-split scan where it beats the one-lane-per-row
// kernels for `L` tokens of rows with `carried` coordinates, else 0.
int rows_scan_lanes(int mode, int carried, long long B, int L, int H, int P, int G);
template <int N8, int N4, int NZ, int MODE>
hipError_t launch_rows(const StepArgs& a, hipStream_t stream);

// Tokens whose records a ridge scan holds at a time: those of 256 MiB, in
// whole dt batches of 64.  A piece costs a trip of the carry through memory and
// two launches: with 128 MiB the second half of 256 tokens at batch 128 took
// 1.3% (24/44/60 5,537 -> 5,608 us), the last 32 of 96 at batch 256 4 to 5%.
inline int64_t ridge_piece(int64_t batch, int64_t G) {
  const int64_t tokens = (256 << 10) / (batch * G);
  return tokens < 64 ? 64 : tokens & ~(int64_t)63;
}

// The same scan of dense 3-bit rows: a.lo the codes, a.s8 the scale pairs,
// a.perm the table.  P % 8 == 0; every array 16-byte aligned.
hipError_t launch_dense3_rows(const StepArgs& a, int equalizer, hipStream_t stream);

}  // namespace m2r
