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

}  // namespace m2r
