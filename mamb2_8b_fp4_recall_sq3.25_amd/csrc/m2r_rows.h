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
// Whether the scan of rows with `carried` coordinates beats the one-lane-per-row
// kernels at these 64-row slots and tokens.
bool rows_scan_pays(int mode, int carried, long long slots, int L);
template <int N8, int N4, int NZ, int MODE>
hipError_t launch_rows(const StepArgs& a, hipStream_t stream);

// The same scan of dense 3-bit rows: a.lo the codes, a.s8 the scale pairs,
// a.perm the table.  P % 8 == 0; every array 16-byte aligned.
hipError_t launch_dense3_rows(const StepArgs& a, int equalizer, hipStream_t stream);

}  // namespace m2r
