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
// tokens on 8 / 4 / 2 / 1 lanes at batches of 128 slots each (records included):
//                     3                 4               6               8
//   ridge 24/44/60    77/ 81/ 98/154  110/ 86/100/155  143/108/115/159  177/129/118/161
//   ridge 8/76/44     78/ 90/121      108/ 94/122      140/118/135      177/164/138
//   tier 32/32/64     48/ 51/ 73/123   62/ 54/ 75/123   88/ 67/ 80/123  108/ 82/ 81/125
//   tier 8/80/40      59/ 74/101       85/ 77/102      110/ 95/112      141/117/115
//   legacy 16/64/48   55/ 64/ 85       79/ 66/ 86      104/ 85/ 97      134/105/ 99
//   dense3            65/ 75/121       98/ 79/122      125/102/132      162/145/135
//                     12               16              32              64
//   ridge 24/44/60   249/177/148/179  321/222/204/185  -/410/344/352   -/791/649/690
//   ridge 8/76/44    251/210/237      323/269/257      -/512/498       -/980/975
//   tier 32/32/64    151/115/105/141  196/149/155/144  -/277/260/279   -/536/485/546
//   tier 8/80/40     206/169/205      267/217/226      -/408/447       -/787/878
//   legacy 16/64/48  193/148/129      253/193/184      -/357/311       -/696/591
//   dense3           235/193/246      309/251/267      -/478/521       -/931/1039
// The first three lines are where the order changes, within 3%, at every width
// (batch 5 and 7 go the way of 6 and 8).  Past 1,024 slots the rule is coarser:
// four lanes are right for 84 and more coordinates (within 5%), one lane for at
// most 72 at 1,792 to 2,048 slots, but two lanes measure 1 to 17% faster than the
// rule's for at most 72 at 1,280 and 1,536 slots, and 2 to 15% for some widths
// beyond (24/44/60 and 32/32/64 from 4,096 slots, 16/60/52 from 1,792, 16/64/48 at
// 1,536 and from 2,048).  One lane has all carried coordinates and updates in
// registers: with more than 72 they spill (8/76/44 at batch 16: 279 against 273
// on four lanes).
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
