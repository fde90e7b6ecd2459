// Attention backward: dQ at head dims 192 and 256 (query-stationary, K/V tiles
// shared by the waves).  At 256 four waves of 16 rows, one per SIMD, cover the
// work item's rows in two passes over its keys (the Q/dO rows and dQ
// accumulators of 32 rows per wave, or of 16 rows at two waves per SIMD, do not
// fit the registers); at 192 32 rows per wave do fit and one pass suffices (8
// sequences of 512 to 2048 rows at 16/8 heads 258 us against 326 in two passes;
// eight waves of 16 rows spill).  Compiled with the default code generation
// (attention_dq.hip compiles the narrower instances with MFMA results in VGPRs).
#include "attention_dq_wave.h"

namespace ts {
namespace attn {

template <typename E, int NQB, int HD, int NP>
void launch_dq_wide_t(const ts_attn_problem& P, int gc, dim3 grid, ts_attn_rows q, ts_attn_rows dout,
                      const float* rowstats, int64_t lse_ld, ts_attn_rows dq, hipStream_t s) {
  ts::TimedLaunch timed_("attention.dq_kernel", s);
  const dim3 block(512 / (NQB * NP));
  if (gc == 4)
    hipLaunchKernelGGL((dq_wave_kernel<E, NQB, HD, 4, NP>), grid, block, 0, s, P, q, dout, rowstats, lse_ld, dq);
  else if (gc == 2)
    hipLaunchKernelGGL((dq_wave_kernel<E, NQB, HD, 2, NP>), grid, block, 0, s, P, q, dout, rowstats, lse_ld, dq);
  else
    hipLaunchKernelGGL((dq_wave_kernel<E, NQB, HD, 1, NP>), grid, block, 0, s, P, q, dout, rowstats, lse_ld, dq);
}

template <typename E>
void launch_dq_wide_e(const ts_attn_problem& P, int gc, dim3 grid, ts_attn_rows q, ts_attn_rows dout,
                      const float* rowstats, int64_t lse_ld, ts_attn_rows dq, hipStream_t s) {
  if (P.head_dim == 192)
    launch_dq_wide_t<E, 2, 192, 1>(P, gc, grid, q, dout, rowstats, lse_ld, dq, s);
  else
    launch_dq_wide_t<E, 1, 256, 2>(P, gc, grid, q, dout, rowstats, lse_ld, dq, s);
}

void launch_dq_wide(const ts_attn_problem& P, int gc, dim3 grid, ts_attn_rows q, ts_attn_rows dout,
                    const float* rowstats, int64_t lse_ld, ts_attn_rows dq, hipStream_t s) {
  if (P.dtype == kF16)
    launch_dq_wide_e<f16>(P, gc, grid, q, dout, rowstats, lse_ld, dq, s);
  else
    launch_dq_wide_e<bf16>(P, gc, grid, q, dout, rowstats, lse_ld, dq, s);
}

}  // namespace attn
}  // namespace ts
