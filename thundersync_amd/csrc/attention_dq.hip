// Attention backward: row statistics and dQ (query-stationary).
#include "attention_dq_wave.h"

namespace ts {
namespace attn {

// ---------------------------------------------------------------------------
// backward preprocess: per (head, row) the pair (lse * log2(e), delta) with
// delta = sum_d dO * O (fp32); a row that saw no key (lse = -inf) gets +inf
// so that exp2(s * scale * log2(e) - lse2) is 0.  The two values of a row are
// adjacent so the backward kernels fetch a tile's statistics in one load.
// ---------------------------------------------------------------------------
template <typename E, int HD>
__global__ __launch_bounds__(kThreads) void delta_kernel(ts_attn_rows O, ts_attn_rows dO,
                                                         const float* __restrict__ lse,
                                                         float* __restrict__ rowstats, int64_t lse_ld,
                                                         int64_t rows, int hq) {
  const int64_t pair = (int64_t)blockIdx.x * (kThreads / 16) + threadIdx.x / 16;
  const int sub = threadIdx.x & 15;
  const int64_t row = pair / hq;
  const int h = (int)(pair % hq);
  if (row >= rows) return;
  // 16 lanes per (row, head), HD / 16 elements each.  O is read only here
  // (non-temporal); dO stays cached for the dQ and dK/dV kernels that follow
  constexpr int PER = HD / 16;
  const bf16* op = (const bf16*)O.ptr + row * O.row_stride + (int64_t)h * O.head_stride + PER * sub;
  const bf16* dp = (const bf16*)dO.ptr + row * dO.row_stride + (int64_t)h * dO.head_stride + PER * sub;
  float acc = 0.f;
  auto add2 = [&](uint32_t a, uint32_t b) {
    acc = fmaf(bits_to_f<E>(a & 0xffffu), bits_to_f<E>(b & 0xffffu), acc);
    acc = fmaf(bits_to_f<E>(a >> 16), bits_to_f<E>(b >> 16), acc);
  };
  if constexpr (PER % 8 == 0) {
#pragma unroll
    for (int c = 0; c < PER / 8; ++c) {
      const u32x4 a = __builtin_nontemporal_load(reinterpret_cast<const u32x4*>(op + 8 * c));
      const u32x4 b = ld16(dp + 8 * c);
#pragma unroll
      for (int i = 0; i < 4; ++i) add2(a[i], b[i]);
    }
  } else {
    // PER = 2, 4 or 6: 4-byte loads
#pragma unroll
    for (int c = 0; c < PER / 2; ++c)
      add2(__builtin_nontemporal_load(reinterpret_cast<const uint32_t*>(op) + c),
           reinterpret_cast<const uint32_t*>(dp)[c]);
  }
#pragma unroll
  for (int msk = 8; msk >= 1; msk >>= 1) acc += shfl_xor(acc, msk);
  if (sub == 0) {
    const int64_t at = (int64_t)h * lse_ld + row;
    const float l = lse[at];
    rowstats[2 * at] = l == neg_inf() ? __builtin_huge_valf() : l * kLog2e;
    rowstats[2 * at + 1] = acc;
  }
}

// ---------------------------------------------------------------------------
// backward dQ (query-stationary)
template <typename E, int HD>
void launch_delta_hd(const ts_attn_problem& P, ts_attn_rows out, ts_attn_rows dout, const float* lse, float* rowstats,
                     int64_t lse_ld, int64_t pairs, hipStream_t s) {
  ts::TimedLaunch timed_("attention.delta_kernel", s);
  hipLaunchKernelGGL((delta_kernel<E, HD>), dim3((unsigned)((pairs + 15) / 16)), dim3(kThreads), 0, s, out, dout, lse,
                     rowstats, lse_ld, P.q_rows, P.hq);
}

template <typename E>
int launch_delta_t(const ts_attn_problem& P, ts_attn_rows out, ts_attn_rows dout, const float* lse,
                 float* rowstats, int64_t lse_ld, hipStream_t s) {
  const int64_t pairs = P.q_rows * P.hq;
  if (pairs == 0) return TS_OK;
  switch (P.head_dim) {
    case 32: launch_delta_hd<E, 32>(P, out, dout, lse, rowstats, lse_ld, pairs, s); break;
    case 64: launch_delta_hd<E, 64>(P, out, dout, lse, rowstats, lse_ld, pairs, s); break;
    case 96: launch_delta_hd<E, 96>(P, out, dout, lse, rowstats, lse_ld, pairs, s); break;
    case 192: launch_delta_hd<E, 192>(P, out, dout, lse, rowstats, lse_ld, pairs, s); break;
    case 256: launch_delta_hd<E, 256>(P, out, dout, lse, rowstats, lse_ld, pairs, s); break;
    default: launch_delta_hd<E, D>(P, out, dout, lse, rowstats, lse_ld, pairs, s);
  }
  return ts::check_launch("ts_attn_bwd (delta)");
}

// query rows per wave of the dQ kernel (16: eight waves, two per SIMD; 32: four)
constexpr int kDqRowsPerWave = 16;

template <typename E, int NQB, int HD>
void launch_dq_hd(const ts_attn_problem& P, int gc, dim3 grid, ts_attn_rows q, ts_attn_rows dout,
                  const float* rowstats, int64_t lse_ld, ts_attn_rows dq, hipStream_t s) {
  ts::TimedLaunch timed_("attention.dq_kernel", s);
  const dim3 block(64 * 8 / NQB);
  if (gc == 4)
    hipLaunchKernelGGL((dq_wave_kernel<E, NQB, HD, 4>), grid, block, 0, s, P, q, dout, rowstats, lse_ld, dq);
  else if (gc == 2)
    hipLaunchKernelGGL((dq_wave_kernel<E, NQB, HD, 2>), grid, block, 0, s, P, q, dout, rowstats, lse_ld, dq);
  else
    hipLaunchKernelGGL((dq_wave_kernel<E, NQB, HD, 1>), grid, block, 0, s, P, q, dout, rowstats, lse_ld, dq);
}

template <typename E>
int launch_dq_t(const ts_attn_problem& P, ts_attn_rows q, ts_attn_rows dout, const float* rowstats,
              int64_t lse_ld, ts_attn_rows dq, hipStream_t s) {
  const int group = P.hq / P.hkv;
  const int gc = heads_per_block(group);
  const dim3 grid((unsigned)(P.n_q_work * P.hkv * (group / gc)));
  switch (P.head_dim) {
    case 32: launch_dq_hd<E, 2, 32>(P, gc, grid, q, dout, rowstats, lse_ld, dq, s); break;
    case 64: launch_dq_hd<E, 2, 64>(P, gc, grid, q, dout, rowstats, lse_ld, dq, s); break;
    case 96: launch_dq_hd<E, 2, 96>(P, gc, grid, q, dout, rowstats, lse_ld, dq, s); break;
    case 192:
    case 256: launch_dq_wide(P, gc, grid, q, dout, rowstats, lse_ld, dq, s); break;
    default: launch_dq_hd<E, kDqRowsPerWave / 16, D>(P, gc, grid, q, dout, rowstats, lse_ld, dq, s);
  }
  return ts::check_launch("ts_attn_bwd (dq)");
}

int launch_delta(const ts_attn_problem& P, ts_attn_rows out, ts_attn_rows dout, const float* lse,
                 float* rowstats, int64_t lse_ld, hipStream_t s) {
  return P.dtype == kF16 ? launch_delta_t<f16>(P, out, dout, lse, rowstats, lse_ld, s)
                         : launch_delta_t<bf16>(P, out, dout, lse, rowstats, lse_ld, s);
}

int launch_dq(const ts_attn_problem& P, ts_attn_rows q, ts_attn_rows dout, const float* rowstats,
              int64_t lse_ld, ts_attn_rows dq, hipStream_t s) {
  return P.dtype == kF16 ? launch_dq_t<f16>(P, q, dout, rowstats, lse_ld, dq, s)
                         : launch_dq_t<bf16>(P, q, dout, rowstats, lse_ld, dq, s);
}

}  // namespace attn
}  // namespace ts
