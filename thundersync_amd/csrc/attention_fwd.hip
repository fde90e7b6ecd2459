// Attention forward kernel (query-stationary online softmax).
#include "attention_impl.h"

namespace ts {
namespace attn {

// ---------------------------------------------------------------------------
// forward with the waves sharing K/V tiles (every head dim and GQA group, GC
// heads per work-group)
//
// A work-group owns 128 / GC query rows of one segment for GC query heads of
// one GQA group; wave w takes head w % GC and 16 NQB rows (at head dim 128
// with GC = 4: NQB = 2, four waves; NQB = 1, eight waves of 16 rows, four
// waves per SIMD, measured no faster on C2 at 1.32 ms; at head dim 256
// NQB = 1, eight waves, two per SIMD, one work-group per CU for its 128 KB of
// tiles).  The heads share K/V tiles of KT keys (32 at head dim 128: 32 KB
// of stages per work-group, three work-groups and three waves per SIMD at 168
// VGPRs, against two with 64-key tiles: C2 forward 1.20 -> 1.09 ms; 32 at 192,
// where 16 rows a wave over 64-key tiles took 172 us against 136 for 8 sequences
// of 512 to 2048 rows at 16/8 heads; 64 at the others: 59 us against 63 with 32 at
// head dim 64 there, 65 with 16 rows a wave), streamed by buffer DMA into
// double-buffered swizzled LDS stages (one work-group barrier per tile).  Q rows
// stay in registers as B operands of S^T = K Q^T; V^T for O^T += V^T P^T comes
// from ds_read_b64_tr_b16.  Per 32 keys of a tile each lane owns one query column
// (16 qb + j16) and 8 of the keys, the others sitting in the lanes j16 + 16, + 32,
// + 48.  The softmax runs in the log2 domain.  Only tiles that cross the diagonal
// or pass a run's end are masked.
//
// The reference point m of a row: at head dims 128 and 256 it moves only when the
// row maximum exceeds it by more than 8 (a factor of 256), so that the
// accumulators are rescaled in the rare tile where that happens (skipped wave-wide
// otherwise), with the scale folded into one FMA per score.  At the other head
// dims it is the running maximum, exactly, of scores already in log2 units: the
// largest weight of a row is 1, which the rounding of the weights to 16 bits
// leaves as it is, and scores and scales of any size and sign keep their softmax.
// Against 64 bits an fp16 cohort at head dim 64 is off by 3.2e-4, by 3.3e-4 with
// the other rule, which takes 49 us there against 64.
//
// Against K/V tiles passed through registers between two barriers (8 sequences of
// 512 to 2048 rows, us): head dim 64 at 16/8 heads 72 -> 64, at 32/8 122 -> 104, 32
// 62 -> 55, 96 93 -> 77, 192 at 24/4 430 -> 184.
// ---------------------------------------------------------------------------
constexpr float kRescaleSlack = 8.f;    // log2 units
constexpr float kRescaleBound = 256.f;  // 2^kRescaleSlack

#ifndef TS_FWD_KT128
#define TS_FWD_KT128 32
#endif
// keys per K/V tile at head dim 128 for GQA groups that are not a multiple of 4
#ifndef TS_FWD_KT128_GC
#define TS_FWD_KT128_GC 32
#endif
// work-groups per CU: their LDS stages (two K/V stages of KT keys) and registers
template <int NQB, int HD, int KT>
constexpr int fwd_occupancy() {
  if (HD < 128 || HD == 192) return HD <= 64 ? 4 : HD == 96 ? 3 : 2;
  return HD > 128 ? (NQB == 1 ? 2 : 1) : (NQB == 1 ? 4 : (KT == 32 ? 3 : 2));
}

// whether the reference point of a row moves only past kRescaleSlack
template <int HD> constexpr bool fwd_lazy_reference() { return HD % 128 == 0; }

// SPLIT: the launch's y blocks are parts of each item's keys (launches whose
// items leave CUs idle, ts_attn_fwd_parts); a part writes its unnormalised fp32
// accumulators and (m, l) per row, which fwd_merge_kernel combines.
template <typename E, int NQB, int HD = D, int GC = 4, int KT = BK, bool SPLIT = false>
__global__ __launch_bounds__(64 * 8 / NQB, (fwd_occupancy<NQB, HD, KT>())) void fwd_wave_kernel(
    ts_attn_problem P, ts_attn_rows Q, ts_attn_rows O, float* __restrict__ lse, int64_t lse_ld,
    PartSums part) {
  constexpr int kWaves = 8 / NQB;
  constexpr int NKS = HD / 32, NMB = HD / 16;  // k-steps of S; 16-column blocks of O
  constexpr bool kLazy = fwd_lazy_reference<HD>();
  static_assert(KT == 64 || KT == 32, "tiles of 64 or 32 keys");
  __shared__ __attribute__((aligned(16))) bf16 s_k0[KT * HD];
  __shared__ __attribute__((aligned(16))) bf16 s_v0[KT * HD];
  __shared__ __attribute__((aligned(16))) bf16 s_k1[KT * HD];
  __shared__ __attribute__((aligned(16))) bf16 s_v1[KT * HD];
  const int tid = threadIdx.x, lane = tid & 63;
  const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
  const int g4 = lane >> 4, j16 = lane & 15;
  int yb;
  const int item = task_of(P.n_q_work, P.n_q_long, yb);
  const int seg_id = uniform_table(P.q_work)[2 * item];
  const int q0 = uniform_table(P.q_work)[2 * item + 1];
  const int group = P.hq / P.hkv;
  const int chunks = group / GC;
  const int hk = yb / chunks;
  const int h = hk * group + (yb % chunks) * GC + (wave % GC);
  const int qw = q0 + 16 * NQB * (wave / GC);  // this wave's first row
  const ts_attn_segment seg = load_uniform(P.segs, seg_id);
  const int T = seg.q_len;
  const int off = seg.kv_len - seg.q_len;
  const int last = min(q0 + 16 * NQB * kWaves / GC, T) - 1;
  const int w_last = min(qw + 16 * NQB, T) - 1;  // this wave's last row
  int begin = 0, stop = off + last + 1;
  if constexpr (SPLIT) part_of<KT>(stop, (int)blockIdx.y, (int)gridDim.y, begin, stop);
  const float c = P.scale * kLog2e;

  // Q rows as B operands: qreg[qb][ks] = row qw + 16 qb + j16, columns 32 ks + 8 g4 ..
  bf16x8 qreg[NQB][NKS];
  load_rows_b<NQB, HD>(qreg, (const bf16*)Q.ptr + (seg.q_row0 + qw) * Q.row_stride + (int64_t)h * Q.head_stride,
              Q.row_stride, T - qw, lane);
  f32x4 acc[NMB][NQB];
  float m[NQB], l[NQB];  // reference point (log2 units) of this lane's column; its part of the
                         // column's sum of exp2(s c - m)
#pragma unroll
  for (int qb = 0; qb < NQB; ++qb) {
#pragma unroll
    for (int mb = 0; mb < NMB; ++mb) acc[mb][qb] = f32x4{0.f, 0.f, 0.f, 0.f};
    m[qb] = neg_inf();
    l[qb] = 0.f;
  }
  int ro[kRowOffsets<HD>], to[2 * kRowOffsets<HD>];
  swizzled_offsets<HD>(lane, ro, to);

  auto step = [&](auto bsel, TileCursor& cur) {
    const int kpos = cur.kpos, run_len = cur.len;
    const int kt0 = cur.kt0;
    const TileCursor nxt = next_kv_tile<KT>(P, seg, hk, stop, cur);
    __builtin_amdgcn_s_waitcnt(0);  // this wave's part of the tile has landed
    __syncthreads();                // every part has, and the other stage is free
    const bf16* tk = bsel.value == 0 ? s_k0 : s_k1;
    const bf16* tv = bsel.value == 0 ? s_v0 : s_v1;
    if (nxt.sp < seg.nspan)
      issue_kv_tile<kWaves, HD, KT>(wave, lane, nxt, bsel.value == 0 ? s_k1 : s_k0, bsel.value == 0 ? s_v1 : s_v0);

    const bool masked = (kpos + kt0 + KT - 1 > off + qw) | (kt0 + KT > run_len);
    // a tile that starts past the wave's last visible key adds nothing: at the
    // narrow head dims it is passed over, so that an infinite or NaN component
    // there (times a weight of 0) stays out of rows that do not see it
    if (HD % 128 != 0 && kpos + kt0 > off + w_last) {
      cur = nxt;
      return;
    }
    // two halves of 32 keys, each one online-softmax update:
    // S^T = K Q^T with sc[kb][qb] holding keys 32 ss + 16 kb + 4 g4 + i of column
    // 16 qb + j16, then O^T += V^T P^T with slot j <-> key 32 ss + 16 (j >> 2) + 4 g4 + (j & 3)
#pragma unroll
    for (int ss = 0; ss < KT / 32; ++ss) {
      f32x4 sc[2][NQB];
      // wave priority 1 over the MFMA phases, 0 over the softmax: of the two
      // waves on a SIMD, the one with MFMAs to issue goes first (fwd -1.4 %)
      __builtin_amdgcn_s_setprio(1);
#pragma unroll
      for (int kb = 0; kb < 2; ++kb) {
#pragma unroll
        for (int qb = 0; qb < NQB; ++qb) sc[kb][qb] = f32x4{0.f, 0.f, 0.f, 0.f};
#pragma unroll
        for (int ks = 0; ks < NKS; ++ks) {
          const bf16x8 ak = as_bf16x8(ld16(tk + ro_of<HD>(ro, ks) + (32 * ss + 16 * kb) * HD));
#pragma unroll
          for (int qb = 0; qb < NQB; ++qb) sc[kb][qb] = mma16<E>(ak, qreg[qb][ks], sc[kb][qb]);
        }
      }
      // K fragment reads three (kb, ks) steps ahead of their MFMAs
      __builtin_amdgcn_sched_group_barrier(0x100, 3, 1);
#pragma unroll
      for (int st = 0; st < 2 * NKS; ++st) {
        __builtin_amdgcn_sched_group_barrier(0x008, NQB, 1);
        if (st + 3 < 2 * NKS) __builtin_amdgcn_sched_group_barrier(0x100, 1, 1);
      }
      __builtin_amdgcn_s_setprio(0);
      // at an exact reference point the scores go to log2 units here, and the
      // largest one of a row to exactly 0 below
      if constexpr (!kLazy) {
#pragma unroll
        for (int kb = 0; kb < 2; ++kb)
#pragma unroll
          for (int qb = 0; qb < NQB; ++qb) sc[kb][qb] *= c;
      }
      if (masked) {
#pragma unroll
        for (int kb = 0; kb < 2; ++kb)
#pragma unroll
          for (int qb = 0; qb < NQB; ++qb) {
            const int key0 = kt0 + 32 * ss + 16 * kb + 4 * g4;  // key of element i = key0 + i
            const int lim = min(off + qw + 16 * qb + j16 - kpos, run_len - 1) - key0;
#pragma unroll
            for (int i = 0; i < 4; ++i)
              if (i > lim) sc[kb][qb][i] = neg_inf();
          }
      }
      float pe[2][NQB][4], ps[NQB];
      auto exponentials = [&](int qb) __attribute__((always_inline)) {
        const float mref = m[qb] == neg_inf() ? 0.f : m[qb];
        ps[qb] = 0.f;
#pragma unroll
        for (int kb = 0; kb < 2; ++kb)
#pragma unroll
          for (int i = 0; i < 4; ++i) {
            pe[kb][qb][i] = fast_exp2(kLazy ? fmaf(sc[kb][qb][i], c, -mref) : sc[kb][qb][i] - mref);
            ps[qb] += pe[kb][qb][i];
          }
      };
      // Fast path: the exponentials against the current reference point m.
      // They stand unless some score exceeds m by more than kRescaleSlack, which
      // a lane detects as a partial sum above 2^kRescaleSlack (every term is
      // positive), or m is still -inf; then, rarely, the half is redone on the
      // slow path: column maxima, the move of m with the rescale of O and the
      // row sum, and the exponentials again.
      bool redo = !kLazy;
      if constexpr (kLazy) {
#pragma unroll
        for (int qb = 0; qb < NQB; ++qb) {
          exponentials(qb);
          redo |= (m[qb] == neg_inf()) | (ps[qb] > kRescaleBound);
        }
      }
      if (!kLazy || __builtin_amdgcn_ballot_w64(redo) != 0) {
#pragma unroll
        for (int qb = 0; qb < NQB; ++qb) {
          float mx = fmaxf(fmaxf(fmaxf(sc[0][qb][0], sc[0][qb][1]), fmaxf(sc[0][qb][2], sc[0][qb][3])),
                           fmaxf(fmaxf(sc[1][qb][0], sc[1][qb][1]), fmaxf(sc[1][qb][2], sc[1][qb][3])));
          mx = rows_max4(mx);
          // maximum in log2 units (-inf if the column sees none of these keys)
          const float mt = kLazy ? mx * c : mx;
          const bool move = mt > m[qb] + (kLazy ? kRescaleSlack : 0.f);
          if (__builtin_amdgcn_ballot_w64(move) != 0) {
            const float mnew = move ? mt : m[qb];
            // 0 on the first finite score (m = -inf); a row whose scores so far are
            // all -inf (or, in a part, none of whose keys it sees) stays as it is beside
            // rows that move
            const float alpha = move ? fast_exp2(m[qb] - mnew) : 1.f;
            l[qb] *= alpha;
#pragma unroll
            for (int mb = 0; mb < NMB; ++mb) acc[mb][qb] *= alpha;
            m[qb] = mnew;
          }
          exponentials(qb);
        }
      }
#pragma unroll
      for (int qb = 0; qb < NQB; ++qb) l[qb] += ps[qb];
      bf16x8 pk[NQB];
#pragma unroll
      for (int qb = 0; qb < NQB; ++qb) {
        float tmp[8];
#pragma unroll
        for (int j = 0; j < 8; ++j) tmp[j] = pe[j >> 2][qb][j & 3];
        pk[qb] = pack8<E>(tmp);
      }
      __builtin_amdgcn_s_setprio(1);
#pragma unroll
      for (int mb = 0; mb < NMB; ++mb) {
        const u32x2 a0 = tr_read(tv + to_of<HD>(to, mb) + 32 * ss * HD);
        const u32x2 a1 = tr_read(tv + to_of<HD>(to, mb) + (32 * ss + 16) * HD);
        const bf16x8 a = as_bf16x8(u32x4{a0[0], a0[1], a1[0], a1[1]});
#pragma unroll
        for (int qb = 0; qb < NQB; ++qb) acc[mb][qb] = mma16<E>(a, pk[qb], acc[mb][qb]);
      }
      // V^T fragment reads kept four blocks ahead of their MFMAs
      __builtin_amdgcn_sched_group_barrier(0x100, 8, 0);
#pragma unroll
      for (int mb = 0; mb < NMB; ++mb) {
        __builtin_amdgcn_sched_group_barrier(0x008, NQB, 0);
        if (mb + 4 < NMB) __builtin_amdgcn_sched_group_barrier(0x100, 2, 0);
      }
      __builtin_amdgcn_sched_barrier(0);
      __builtin_amdgcn_s_setprio(0);
    }
    cur = nxt;
  };

  TileCursor cur = SPLIT ? first_kv_tile_from<KT>(P, seg, hk, begin, stop) : first_kv_tile<KT>(P, seg, hk, stop);
  if (cur.sp < seg.nspan) issue_kv_tile<kWaves, HD, KT>(wave, lane, cur, s_k0, s_v0);
  while (cur.sp < seg.nspan) {
    step(std::integral_constant<int, 0>{}, cur);
    if (cur.sp >= seg.nspan) break;
    step(std::integral_constant<int, 1>{}, cur);
  }

  // O = acc / l; acc[mb][qb] lane holds d = 16 mb + 4 g4 + i of row qw + 16 qb + j16
#pragma unroll
  for (int qb = 0; qb < NQB; ++qb) {
    const float ls = rows_sum4(l[qb]);
    const int row = qw + 16 * qb + j16;
    if (row >= T) continue;
    if constexpr (SPLIT) {
      const int64_t at = part_row<128>(P, part, (int)blockIdx.y, item * P.hkv * chunks + yb,
                                       (row - q0) * GC + wave % GC, h, seg.q_row0 + row);
      float* prow = part.ptr + at * HD + 4 * g4;
#pragma unroll
      for (int mb = 0; mb < NMB; ++mb) *reinterpret_cast<f32x4*>(prow + 16 * mb) = acc[mb][qb];
      if (g4 == 0) {
        float* st = part_stats<HD>(part, (int)gridDim.y) + 2 * at;
        st[0] = m[qb];
        st[1] = ls;
      }
      continue;
    }
    const float inv = ls > 0.f ? 1.f / ls : 0.f;
    bf16* orow = (bf16*)O.ptr + (seg.q_row0 + row) * O.row_stride + (int64_t)h * O.head_stride + 4 * g4;
#pragma unroll
    for (int mb = 0; mb < NMB; ++mb) {
      const f32x4 v = acc[mb][qb] * inv;
      *reinterpret_cast<u32x2*>(orow + 16 * mb) = u32x2{pack2<E>(v[0], v[1]), pack2<E>(v[2], v[3])};
    }
    if (g4 == 0)
      lse[(int64_t)h * lse_ld + seg.q_row0 + row] = ls > 0.f ? (m[qb] + fast_log2(ls)) * kLn2 : neg_inf();
  }
}

// Out and log-sum-exp of a split launch: with M the largest part's m, O =
// sum_p acc_p 2^(m_p - M) / sum_p l_p 2^(m_p - M), the parts in order.  A wave
// takes one (row, head) at a time, HD / 64 consecutive columns a lane; the y
// blocks cut an item's rows and heads so that few items still fill the CUs.
template <typename E, int HD, int GC>
__global__ __launch_bounds__(kThreads) void fwd_merge_kernel(ts_attn_problem P, ts_attn_rows O,
                                                             float* __restrict__ lse, int64_t lse_ld,
                                                             PartSums part, int parts) {
  constexpr int NC = HD / 64;  // columns per lane (2 or 4)
  const int lane = threadIdx.x & 63, wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
  const int chunks = P.hq / P.hkv / GC;
  const int heads = P.hkv * chunks;  // head chunks of an item
  const int item = (int)blockIdx.x / heads, yb = (int)blockIdx.x % heads;
  const int seg_id = uniform_table(P.q_work)[2 * item];
  const int q0 = uniform_table(P.q_work)[2 * item + 1];
  const ts_attn_segment seg = load_uniform(P.segs, seg_id);
  const float* stats = part_stats<HD>(part, parts);
  constexpr int kPairs = 128 / kMergeBlocks;  // (row, head) pairs of a work-group
#pragma unroll 1
  for (int i = wave; i < kPairs; i += kThreads / 64) {
    const int pair = (int)blockIdx.y * kPairs + i;
    const int row = q0 + pair / GC, h = yb * GC + pair % GC;
    if (row >= seg.q_len) break;
    const int64_t at = part_row<128>(P, part, 0, (int)blockIdx.x, pair, h, seg.q_row0 + row), step = part.rows;
    float M = neg_inf();
    for (int p = 0; p < parts; ++p) M = fmaxf(M, stats[2 * (at + p * step)]);
    const float ref = M == neg_inf() ? 0.f : M;
    float acc[NC], L = 0.f;
#pragma unroll
    for (int c = 0; c < NC; ++c) acc[c] = 0.f;
#pragma unroll 4
    for (int p = 0; p < parts; ++p) {
      const float w = fast_exp2(stats[2 * (at + p * step)] - ref);
      L = fmaf(stats[2 * (at + p * step) + 1], w, L);
      const float* x = part.ptr + (at + p * step) * HD + NC * lane;
#pragma unroll
      for (int c = 0; c < NC; ++c) acc[c] = fmaf(x[c], w, acc[c]);
    }
    const float inv = L > 0.f ? 1.f / L : 0.f;
    uint32_t* o = reinterpret_cast<uint32_t*>((bf16*)O.ptr + (seg.q_row0 + row) * O.row_stride +
                                              (int64_t)h * O.head_stride + NC * lane);
#pragma unroll
    for (int c = 0; c < NC; c += 2) o[c / 2] = pack2<E>(acc[c] * inv, acc[c + 1] * inv);
    if (lane == 0) lse[(int64_t)h * lse_ld + seg.q_row0 + row] = L > 0.f ? (M + fast_log2(L)) * kLn2 : neg_inf();
  }
}

// query rows per wave of the forward kernel (32: four waves per work-group; 16: eight)
constexpr int kFwdRowsPerWave = 32;

// whole items, or parts of them (head dims 128 and 256)
template <typename E, int NQB, int HD, int GC, int KT>
void launch_fwd_wave(const ts_attn_problem& P, dim3 grid, ts_attn_rows q, ts_attn_rows out, float* lse, int64_t lse_ld,
                     int parts, PartSums part, hipStream_t s) {
  if (parts <= 1) {
    ts::TimedLaunch timed_("attention.fwd_kernel", s);
    hipLaunchKernelGGL((fwd_wave_kernel<E, NQB, HD, GC, KT>), grid, dim3(64 * 8 / NQB), 0, s, P, q, out, lse, lse_ld,
                       part);
    return;
  }
  if constexpr (HD % 128 == 0) {
    {
      ts::TimedLaunch timed_("attention.fwd_kernel", s);
      hipLaunchKernelGGL((fwd_wave_kernel<E, NQB, HD, GC, KT, true>), dim3(grid.x, parts), dim3(64 * 8 / NQB), 0, s, P,
                         q, out, lse, lse_ld, part);
    }
    ts::TimedLaunch timed_("attention.fwd_merge_kernel", s);
    hipLaunchKernelGGL((fwd_merge_kernel<E, HD, GC>), dim3(grid.x, kMergeBlocks), dim3(kThreads), 0, s, P, out, lse,
                       lse_ld, part, parts);
  }
}

template <typename E, int NQB, int HD, int KT>
void launch_fwd_hd(const ts_attn_problem& P, int gc, dim3 grid, ts_attn_rows q, ts_attn_rows out, float* lse,
                   int64_t lse_ld, int parts, PartSums part, hipStream_t s) {
  if (gc == 4) launch_fwd_wave<E, NQB, HD, 4, KT>(P, grid, q, out, lse, lse_ld, parts, part, s);
  else if (gc == 2) launch_fwd_wave<E, NQB, HD, 2, KT>(P, grid, q, out, lse, lse_ld, parts, part, s);
  else launch_fwd_wave<E, NQB, HD, 1, KT>(P, grid, q, out, lse, lse_ld, parts, part, s);
}

template <typename E>
int launch_fwd_t(const ts_attn_problem& P, ts_attn_rows q, ts_attn_rows out, float* lse, int64_t lse_ld, int parts,
                 PartSums part, hipStream_t s) {
  const int group = P.hq / P.hkv;
  const int gc = heads_per_block(group);
  const dim3 grid((unsigned)(P.n_q_work * P.hkv * (group / gc)));
  switch (P.head_dim) {
    case 32: launch_fwd_hd<E, 2, 32, BK>(P, gc, grid, q, out, lse, lse_ld, parts, part, s); break;
    case 64: launch_fwd_hd<E, 2, 64, BK>(P, gc, grid, q, out, lse, lse_ld, parts, part, s); break;
    case 96: launch_fwd_hd<E, 2, 96, BK>(P, gc, grid, q, out, lse, lse_ld, parts, part, s); break;
    case 192: launch_fwd_hd<E, 2, 192, 32>(P, gc, grid, q, out, lse, lse_ld, parts, part, s); break;
    case 256: launch_fwd_hd<E, 1, 256, BK>(P, gc, grid, q, out, lse, lse_ld, parts, part, s); break;
    default: {
      constexpr int NQB = kFwdRowsPerWave / 16;
      if (gc == 4) launch_fwd_wave<E, NQB, D, 4, TS_FWD_KT128>(P, grid, q, out, lse, lse_ld, parts, part, s);
      else if (gc == 2) launch_fwd_wave<E, 2, D, 2, TS_FWD_KT128_GC>(P, grid, q, out, lse, lse_ld, parts, part, s);
      else launch_fwd_wave<E, 2, D, 1, TS_FWD_KT128_GC>(P, grid, q, out, lse, lse_ld, parts, part, s);
    }
  }
  return ts::check_launch("ts_attn_fwd");
}

int launch_fwd(const ts_attn_problem& P, ts_attn_rows q, ts_attn_rows out, float* lse, int64_t lse_ld, int parts,
               PartSums part, hipStream_t s) {
  return P.dtype == kF16 ? launch_fwd_t<f16>(P, q, out, lse, lse_ld, parts, part, s)
                         : launch_fwd_t<bf16>(P, q, out, lse, lse_ld, parts, part, s);
}

}  // namespace attn
}  // namespace ts
