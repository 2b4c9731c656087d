// The row-split multi-token scan of ridge-latent rows (m2r_rows_kernel.h),
// behind the kernel that writes its token records, a piece of the tokens at a
// time: the codes between pieces are the ones between tokens.
#include "m2r_rows_kernel.h"
#include "m2r_rows.h"

#include <algorithm>

namespace m2r {

template <int N8, int N4, int NZ, int MODE>
hipError_t launch_rows(const StepArgs& a, hipStream_t stream) {
  const int piece = (int)ridge_piece(a.B, a.G);
  for (int first = 0; first < a.L; first += piece) {
    const int tokens = std::min(piece, a.L - first);
    StepArgs p = a;   // its tokens are the first of each batch row from these pointers on
    p.x += (size_t)first * a.H * a.P;
    p.y += (size_t)first * a.H * a.P;
    p.dt += (size_t)first * a.H;
    p.Bm += (size_t)first * a.G * 128;
    p.Cm += (size_t)first * a.G * 128;
    hipLaunchKernelGGL((k_token_records<N8, N4, NZ>), dim3((tokens + REC_TOKENS - 1) / REC_TOKENS, a.G, a.B), dim3(256),
                       0, stream, p, (float*)a.rec, tokens);
    if (hipError_t e = launch_rows_scan<N8, N4, NZ, MODE>(p, 0, tokens, stream)) return e;
  }
  return hipSuccess;
}
template hipError_t launch_rows<36, 20, 72, MODE_RIDGE>(const StepArgs&, hipStream_t);
template hipError_t launch_rows<16, 60, 52, MODE_RIDGE>(const StepArgs&, hipStream_t);
template hipError_t launch_rows<32, 28, 68, MODE_RIDGE>(const StepArgs&, hipStream_t);
template hipError_t launch_rows<40, 12, 76, MODE_RIDGE>(const StepArgs&, hipStream_t);
template hipError_t launch_rows<24, 44, 60, MODE_RIDGE>(const StepArgs&, hipStream_t);
template hipError_t launch_rows<8, 76, 44, MODE_RIDGE>(const StepArgs&, hipStream_t);
template hipError_t launch_rows<44, 4, 80, MODE_RIDGE>(const StepArgs&, hipStream_t);

}  // namespace m2r
