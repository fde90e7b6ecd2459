// Fused chunked-vocab logprob / entropy of fp32 hidden states and head, on
// the fp32 matrix instruction (v_mfma_f32_32x32x2_f32: fp32 operands and fp32
// FMAs, no operand rounding, 256 FLOP per CU and clock).
//
// Reference: accel/fused_logprob.py:27-58, :137-193, :250-306 for fp32 inputs.
// One tile product serves every kernel: a work-group of four waves forms a
// 64 MI x 64 NJ tile of C(m, n) = sum_k A(m, k) B(k, n), wave (wm, wn) a
// 32 MI x 32 NJ part of it, over operands given by element strides.  K runs
// 32 at a time through two LDS stages: the next stage's global loads are in
// flight in registers while this stage's MFMAs run, one barrier per stage.
// An operand with unit K stride is staged as [rows][32 k] (rows of 36 words: a
// lane reads its row's four k values of four MFMAs as one 16-byte read, and
// the 16 rows of a read pass start in 16 distinct bank groups), any other as
// [32 k][rows] (pitches of 136 and 72 words, = 8 mod 32, put the two lane
// halves, four k rows apart, on distinct halves of the banks).  Either way
// lane half h takes k = 8 g + 4 h + s in MFMA s of group g, for A and B alike.
//
// What bounds it: the MFMA pipes.  A 128 x 128 tile does 64 MFMAs of 64 cycles
// per wave and stage on 32 KB of operands, 8 bytes per CU clock from L2, and
// two work-groups share a CU (74 KB of LDS each) so that one's barrier and
// epilogue run beside the other's MFMAs.  Measured at 2048 rows, hidden 1024,
// vocabulary 32000 with a trainable head, against the vector-ALU tiles of
// logprob_exact.hip: forward 3.72 -> 1.07 ms, dlogits 1.57 -> 0.58 ms per 1024
// rows (115 TFLOP/s), grad_hidden and grad_weight 3.72 -> 0.52 (in 8
// contraction ranges) and 0.62 ms (a library product reaches 148 TFLOP/s);
// grad_hidden's error against 64 bits 3.2e-6 -> 1.1e-6 (shorter sums).
#include <algorithm>
#include <cmath>

#include "gemm_core.h"
#include "logprob_f32.h"
#include "timing.h"
#include "../../include/thundersync_hip.h"

namespace ts {
namespace lpf {

constexpr int BKF = 32;         // K per stage
constexpr int kThreads = 256;   // four waves
constexpr int kSlots = 512;     // work-groups the device holds at once (two per CU)

__device__ __forceinline__ float neg_inf() { return -__builtin_huge_valf(); }

// LDS words of one operand stage of R rows
template <int R, bool KF> constexpr int stage_words() { return KF ? R * 36 : BKF * (R + 8); }

// One operand's tile: R rows (M or N index) x 32 k of x[r sr + k sk].
template <int R, bool KF, bool VEC>
struct Operand {
  static constexpr int NV = R / 32;       // float4 per thread and stage
  static constexpr int PITCH = KF ? 36 : R + 8;
  const float* base;  // row r0, k 0
  int64_t sr, sk;
  int rows;           // valid rows from r0, at least 1
  int64_t K;
  const float* at[NV];  // the vectors of the next whole stage
  f32x4 v[NV];

  __device__ __forceinline__ void init(const float* x, int64_t sr_, int64_t sk_, int64_t r0, int64_t total, int64_t K_,
                                       int64_t k_begin = 0) {
    base = x + r0 * sr_;
    sr = sr_;
    sk = sk_;
    rows = (int)min((int64_t)R, total - r0);
    K = K_;
#pragma unroll
    for (int u = 0; u < NV; ++u)
      at[u] = base + min(row_of(u, threadIdx.x), rows - 1) * sr + (k_begin + k_of(u, threadIdx.x)) * sk;
  }
  // first row and first k of vector u (the four lie along k when KF, along the rows otherwise)
  static __device__ __forceinline__ int row_of(int u, int tid) {
    const int i = u * kThreads + tid;
    return KF ? i / 8 : (i % (R / 4)) * 4;
  }
  static __device__ __forceinline__ int k_of(int u, int tid) {
    const int i = u * kThreads + tid;
    return KF ? (i % 8) * 4 : i / (R / 4);
  }
  // global -> registers, k0 .. k0 + 31 (the stages in order).  Rows past the operand read its last
  // row (their products are discarded); k past K reads as zero.  Whole stages
  // of 16-byte aligned operands take unconditional 16-byte loads.
  __device__ __forceinline__ void load(int64_t k0, int tid) {
    if (VEC && k0 + BKF <= K && (KF || rows == R)) {
#pragma unroll
      for (int u = 0; u < NV; ++u) {
        v[u] = *reinterpret_cast<const f32x4*>(at[u]);
        at[u] += BKF * sk;
      }
    } else {
#pragma unroll
      for (int u = 0; u < NV; ++u)
#pragma unroll
        for (int e = 0; e < 4; ++e) {
          const int r = min(row_of(u, tid) + (KF ? 0 : e), rows - 1);
          const int64_t k = k0 + k_of(u, tid) + (KF ? e : 0);
          v[u][e] = k < K ? base[r * sr + k * sk] : 0.f;
        }
    }
  }
  __device__ __forceinline__ void store(float* lds, int tid) const {
#pragma unroll
    for (int u = 0; u < NV; ++u)
      *reinterpret_cast<f32x4*>(lds + (KF ? row_of(u, tid) * PITCH + k_of(u, tid)
                                          : k_of(u, tid) * PITCH + row_of(u, tid))) = v[u];
  }
  // the four k values k = 8 g + 4 h + s of the lane's row in the 32-row block at row0
  static __device__ __forceinline__ f32x4 frag(const float* lds, int row0, int g, int lane) {
    const int r = row0 + (lane & 31), k = 8 * g + 4 * (lane >> 5);
    if constexpr (KF) {
      return *reinterpret_cast<const f32x4*>(lds + r * PITCH + k);
    } else {
      f32x4 x;
#pragma unroll
      for (int s = 0; s < 4; ++s) x[s] = lds[(k + s) * PITCH + r];
      return x;
    }
  }
};

// acc[mi][nj]: the wave's 32 x 32 blocks; lane l holds column l & 31 and rows
// 8 (i >> 2) + 4 (l >> 5) + (i & 3), i = 0..15.  Starts and ends with the LDS free.
template <int MI, int NJ, class OA, class OB>
__device__ __forceinline__ void tile_product(f32x16 (&acc)[MI][NJ], OA& a, OB& b, int64_t k_begin, int64_t k_end,
                                             float* sa0, float* sb0, float* sa1, float* sb1) {
  const int tid = threadIdx.x, lane = tid & 63, wave = tid >> 6;
  const int wm = wave & 1, wn = wave >> 1;
#pragma unroll
  for (int mi = 0; mi < MI; ++mi)
#pragma unroll
    for (int nj = 0; nj < NJ; ++nj)
#pragma unroll
      for (int i = 0; i < 16; ++i) acc[mi][nj][i] = 0.f;
  if (k_begin >= k_end) return;
  a.load(k_begin, tid);
  b.load(k_begin, tid);
  a.store(sa0, tid);
  b.store(sb0, tid);
  __syncthreads();
  auto stage = [&](const float* sa, const float* sb, float* na, float* nb, int64_t k0) {
    const bool more = k0 + BKF < k_end;
    if (more) {
      a.load(k0 + BKF, tid);
      b.load(k0 + BKF, tid);
    }
#pragma unroll
    for (int g = 0; g < BKF / 8; ++g) {
      f32x4 af[MI], bf[NJ];
#pragma unroll
      for (int mi = 0; mi < MI; ++mi) af[mi] = OA::frag(sa, 32 * (MI * wm + mi), g, lane);
#pragma unroll
      for (int nj = 0; nj < NJ; ++nj) bf[nj] = OB::frag(sb, 32 * (NJ * wn + nj), g, lane);
#pragma unroll
      for (int s = 0; s < 4; ++s)
#pragma unroll
        for (int mi = 0; mi < MI; ++mi)
#pragma unroll
          for (int nj = 0; nj < NJ; ++nj)
            acc[mi][nj] = __builtin_amdgcn_mfma_f32_32x32x2f32(af[mi][s], bf[nj][s], acc[mi][nj], 0, 0, 0);
    }
    if (more) {
      a.store(na, tid);
      b.store(nb, tid);
    }
    __syncthreads();
  };
  for (int64_t k0 = k_begin; k0 < k_end; k0 += 2 * BKF) {
    stage(sa0, sb0, sa1, sb1, k0);
    if (k0 + BKF < k_end) stage(sa1, sb1, sa0, sb0, k0 + BKF);
  }
}

// the row within the tile's 32-row block of accumulator element i
__device__ __forceinline__ int acc_row(int i, int lane) { return 8 * (i >> 2) + 4 * (lane >> 5) + (i & 3); }

#define LPF_STAGES(RA, KFA, RB, KFB)                                                 \
  __shared__ __attribute__((aligned(16))) float sa0[stage_words<RA, KFA>()];         \
  __shared__ __attribute__((aligned(16))) float sb0[stage_words<RB, KFB>()];         \
  __shared__ __attribute__((aligned(16))) float sa1[stage_words<RA, KFA>()];         \
  __shared__ __attribute__((aligned(16))) float sb1[stage_words<RB, KFB>()];

// (max, sum exp(l - max), sum exp(l - max) (l - max)) of two disjoint sets of
// logits.  A set whose maximum is -inf adds only its sums: both 0 when it is
// empty, the third NaN when it holds logits of -inf (0 * -inf, as in the plain
// sum), both NaN when it holds a NaN, which no maximum shows.
__device__ __forceinline__ void merge_stats(float& m, float& s, float& e, float mo, float so, float eo) {
  if (mo == neg_inf()) {
    s += so;
    e += eo;
    return;
  }
  if (m == neg_inf()) {
    m = mo;
    s += so;
    e += eo;
    return;
  }
  const float mn = m > mo ? m : mo;
  const float ca = expf(m - mn), cb = expf(mo - mn);
  e = ca * (e + s * (m - mn)) + cb * (eo + so * (mo - mn));
  s = ca * s + cb * so;
  m = mn;
}

// partial[(3 g + c) rows + r]: row r's statistics c (max, sum, sum (l - max))
// over the vocabulary tiles g, g + G, ...  Tile rows are vocabulary entries,
// tile columns tokens, so each lane keeps the running statistics of its NJ
// tokens in registers over all its tiles; the lane halves and the two
// vocabulary waves meet once at the end.
template <int NJ, bool VEC>
__global__ __launch_bounds__(kThreads, 2) void fwd_stats_kernel(const float* __restrict__ h, int64_t ld_h,
                                                                const float* __restrict__ w, int64_t ld_w,
                                                                int64_t rows, int64_t dim, int64_t vocab, int groups,
                                                                int tok_tiles, float* __restrict__ partial) {
  LPF_STAGES(128, true, 64 * NJ, true)
  const int lane = threadIdx.x & 63, wave = threadIdx.x >> 6;
  const int wm = wave & 1, wn = wave >> 1;
  // the token tiles of a vocabulary group run together on one XCD and share its W rows in L2
  const int id = gemm::xcd_logical(blockIdx.x, groups * tok_tiles);
  const int g = id / tok_tiles;
  const int64_t n0 = (int64_t)(id - g * tok_tiles) * (64 * NJ);
  const int64_t n_tiles = (vocab + 127) / 128;
  float sm[NJ], ss[NJ], se[NJ];
#pragma unroll
  for (int nj = 0; nj < NJ; ++nj) {
    sm[nj] = neg_inf();
    ss[nj] = 0.f;
    se[nj] = 0.f;
  }
  for (int64_t vt = g; vt < n_tiles; vt += groups) {
    f32x16 acc[2][NJ];
    Operand<128, true, VEC> a;
    Operand<64 * NJ, true, VEC> b;
    a.init(w, ld_w, 1, vt * 128, vocab, dim);
    b.init(h, ld_h, 1, n0, rows, dim);
    tile_product<2, NJ>(acc, a, b, 0, dim, sa0, sb0, sa1, sb1);
    const int left = (int)min((int64_t)128, vocab - vt * 128);  // vocabulary entries of the tile
#pragma unroll
    for (int nj = 0; nj < NJ; ++nj) {
      float mx = neg_inf();
      bool any = false;
#pragma unroll
      for (int mi = 0; mi < 2; ++mi)
#pragma unroll
        for (int i = 0; i < 16; ++i)
          if (64 * wm + 32 * mi + acc_row(i, lane) < left) {
            mx = acc[mi][nj][i] > mx ? acc[mi][nj][i] : mx;
            any = true;
          }
      float s = 0.f, e = any && mx == neg_inf() ? __builtin_nanf("") : 0.f;
      if (mx != neg_inf()) {
#pragma unroll
        for (int mi = 0; mi < 2; ++mi)
#pragma unroll
          for (int i = 0; i < 16; ++i)
            if (64 * wm + 32 * mi + acc_row(i, lane) < left) {
              const float x = acc[mi][nj][i] - mx;
              const float p = expf(x);
              s += p;
              e += p * x;
            }
      } else if (any) {
#pragma unroll
        for (int mi = 0; mi < 2; ++mi)
#pragma unroll
          for (int i = 0; i < 16; ++i)
            if (64 * wm + 32 * mi + acc_row(i, lane) < left && acc[mi][nj][i] != neg_inf()) s = __builtin_nanf("");
      }
      merge_stats(sm[nj], ss[nj], se[nj], mx, s, e);
    }
  }
  // lane ^ 32 holds the other rows of the same token; then the wm = 1 waves' tokens through LDS
  float* x = sa0;  // [3][64 NJ]
#pragma unroll
  for (int nj = 0; nj < NJ; ++nj) {
    const float mo = shfl_xor(sm[nj], 32), so = shfl_xor(ss[nj], 32), eo = shfl_xor(se[nj], 32);
    merge_stats(sm[nj], ss[nj], se[nj], mo, so, eo);
    const int col = 32 * (NJ * wn + nj) + (lane & 31);
    if (wm == 1 && lane < 32) {
      x[col] = sm[nj];
      x[64 * NJ + col] = ss[nj];
      x[128 * NJ + col] = se[nj];
    }
  }
  __syncthreads();
  if (wm != 0 || lane >= 32) return;
#pragma unroll
  for (int nj = 0; nj < NJ; ++nj) {
    const int col = 32 * (NJ * wn + nj) + lane;
    merge_stats(sm[nj], ss[nj], se[nj], x[col], x[64 * NJ + col], x[128 * NJ + col]);
    const int64_t r = n0 + col;
    if (r < rows) {
      partial[(3 * (int64_t)g + 0) * rows + r] = sm[nj];
      partial[(3 * (int64_t)g + 1) * rows + r] = ss[nj];
      partial[(3 * (int64_t)g + 2) * rows + r] = se[nj];
    }
  }
}

// one wave per row: merge the G partials, then the target logit as a dot
// product; logprob = l_t - lse (NaN for a target outside the vocabulary),
// entropy = log S - E / S
__global__ __launch_bounds__(kThreads) void combine_kernel(const float* __restrict__ partial, int groups,
                                                           const float* __restrict__ h, int64_t ld_h,
                                                           const float* __restrict__ w, int64_t ld_w,
                                                           const int64_t* __restrict__ target, int64_t rows,
                                                           int64_t dim, int64_t vocab, float* __restrict__ logprob,
                                                           float* __restrict__ entropy, float* __restrict__ lse) {
  const int lane = threadIdx.x & 63;
  const int64_t r = (int64_t)blockIdx.x * (kThreads / 64) + (threadIdx.x >> 6);
  if (r >= rows) return;
  float m = neg_inf(), s = 0.f, e = 0.f;
  for (int g = lane; g < groups; g += 64)
    merge_stats(m, s, e, partial[(3 * (int64_t)g + 0) * rows + r], partial[(3 * (int64_t)g + 1) * rows + r],
                partial[(3 * (int64_t)g + 2) * rows + r]);
#pragma unroll
  for (int o = 1; o < 64; o <<= 1) {
    const float mo = shfl_xor(m, o), so = shfl_xor(s, o), eo = shfl_xor(e, o);
    merge_stats(m, s, e, mo, so, eo);
  }
  const int64_t t = target[r];
  const bool valid = t >= 0 && t < vocab;
  float dot = 0.f;
  if (valid)
    for (int64_t d = lane; d < dim; d += 64) dot = fmaf(h[r * ld_h + d], w[t * ld_w + d], dot);
  dot = wave_sum(dot);
  if (lane == 0) {
    const float l = m + logf(s);
    lse[r] = l;
    logprob[r] = valid ? dot - l : __builtin_nanf("");
    if (entropy) entropy[r] = logf(s) - e / s;
  }
}

// dlogits block [rows, vocab] (row stride ld_dl): -p (g_lp + g_H (log p + H))
// + g_lp [v == t], p = exp(l - lse); g_ent null: the logprob-only objective.
// Tile rows are tokens, tile columns vocabulary entries: a store instruction
// writes 128 consecutive bytes of two rows.
template <int MI, bool VEC>
__global__ __launch_bounds__(kThreads, 2) void dlogits_kernel(const float* __restrict__ h, int64_t ld_h,
                                                              const float* __restrict__ w, int64_t ld_w,
                                                              const int64_t* __restrict__ target,
                                                              const float* __restrict__ lse,
                                                              const float* __restrict__ ent,
                                                              const float* __restrict__ g_lp,
                                                              const float* __restrict__ g_ent, int64_t rows,
                                                              int64_t dim, int64_t vocab, float* __restrict__ dl,
                                                              int64_t ld_dl, int tok_tiles, int v_tiles) {
  LPF_STAGES(64 * MI, true, 128, true)
  const int lane = threadIdx.x & 63, wave = threadIdx.x >> 6;
  const int wm = wave & 1, wn = wave >> 1;
  const int id = gemm::xcd_logical(blockIdx.x, tok_tiles * v_tiles);
  const int64_t n0 = (int64_t)(id / tok_tiles) * 128, m0 = (int64_t)(id % tok_tiles) * (64 * MI);
  f32x16 acc[MI][2];
  Operand<64 * MI, true, VEC> a;
  Operand<128, true, VEC> b;
  a.init(h, ld_h, 1, m0, rows, dim);
  b.init(w, ld_w, 1, n0, vocab, dim);
  tile_product<MI, 2>(acc, a, b, 0, dim, sa0, sb0, sa1, sb1);
#pragma unroll
  for (int mi = 0; mi < MI; ++mi)
#pragma unroll
    for (int i = 0; i < 16; ++i) {
      const int64_t r = m0 + 32 * (MI * wm + mi) + acc_row(i, lane);
      if (r >= rows) continue;
      const float l0 = lse[r], g = g_lp[r];
      const float ge = g_ent ? g_ent[r] : 0.f, hr = g_ent ? ent[r] : 0.f;
      const int64_t t = target[r];
#pragma unroll
      for (int nj = 0; nj < 2; ++nj) {
        const int64_t v = n0 + 32 * (2 * wn + nj) + (lane & 31);
        if (v >= vocab) continue;
        const float lp = acc[mi][nj][i] - l0;  // log p
        const float p = expf(lp);
        float d = -p * (g_ent ? g + ge * (lp + hr) : g);
        if (v == t) d += g;
        dl[r * ld_dl + v] = d;
      }
    }
}

// C [M, N] (row stride ldc) = (or +=) A . B over k ranges of `kper`: with one
// range the tile goes to C, with several each range writes its partial sums
// part[range][M][N] and reduce_kernel adds them in range order.
template <int MI, bool KFA, bool KFB, bool VEC>
__global__ __launch_bounds__(kThreads, 2) void matmul_kernel(const float* __restrict__ a, int64_t a_m, int64_t a_k,
                                                             const float* __restrict__ b, int64_t b_k, int64_t b_n,
                                                             int64_t M, int64_t N, int64_t K, float* __restrict__ c,
                                                             int64_t ldc, int accumulate, int m_tiles, int n_tiles,
                                                             int ranges, int64_t kper, float* __restrict__ part) {
  LPF_STAGES(64 * MI, KFA, 128, KFB)
  const int lane = threadIdx.x & 63, wave = threadIdx.x >> 6;
  const int wm = wave & 1, wn = wave >> 1;
  const int tiles = m_tiles * n_tiles;
  const int id = gemm::xcd_logical(blockIdx.x, tiles * ranges);
  const int ks = id / tiles;
  int mt, nt;
  gemm::grouped_tile(id - ks * tiles, m_tiles, n_tiles, mt, nt);
  const int64_t m0 = (int64_t)mt * (64 * MI), n0 = (int64_t)nt * 128;
  const int64_t kb = ks * kper, ke = min(K, kb + kper);
  f32x16 acc[MI][2];
  Operand<64 * MI, KFA, VEC> oa;
  Operand<128, KFB, VEC> ob;
  oa.init(a, a_m, a_k, m0, M, ke, kb);
  ob.init(b, b_n, b_k, n0, N, ke, kb);
  tile_product<MI, 2>(acc, oa, ob, kb, ke, sa0, sb0, sa1, sb1);
  float* out = ranges > 1 ? part + (int64_t)ks * M * N : c;
  const int64_t ldo = ranges > 1 ? N : ldc;
  const bool add = accumulate && ranges == 1;
#pragma unroll
  for (int mi = 0; mi < MI; ++mi)
#pragma unroll
    for (int i = 0; i < 16; ++i) {
      const int64_t m = m0 + 32 * (MI * wm + mi) + acc_row(i, lane);
      if (m >= M) continue;
#pragma unroll
      for (int nj = 0; nj < 2; ++nj) {
        const int64_t n = n0 + 32 * (2 * wn + nj) + (lane & 31);
        if (n >= N) continue;
        float* p = out + m * ldo + n;
        *p = add ? *p + acc[mi][nj][i] : acc[mi][nj][i];
      }
    }
}

__global__ __launch_bounds__(kThreads) void reduce_kernel(const float* __restrict__ part, int ranges, int64_t M,
                                                          int64_t N, float* __restrict__ c, int64_t ldc,
                                                          int accumulate) {
  const int64_t e = (int64_t)blockIdx.x * kThreads + threadIdx.x;
  if (e >= M * N) return;
  float s = part[e];
  for (int r = 1; r < ranges; ++r) s += part[(int64_t)r * M * N + e];
  float* p = c + e / N * ldc + e % N;
  *p = accumulate ? *p + s : s;
}

// ---------------------------------------------------------------------------
// host side
// ---------------------------------------------------------------------------
bool vec_ok(const float* p, int64_t row_stride) { return (uintptr_t)p % 16 == 0 && row_stride % 4 == 0; }
int64_t tiles_of(int64_t n, int64_t t) { return (n + t - 1) / t; }

// 64-token tiles where the rows fit one, or where 128-token tiles over every
// vocabulary tile would leave some of the device's work-group slots empty
bool narrow(int64_t rows, int64_t vocab) {
  return rows <= 64 || tiles_of(rows, 128) * tiles_of(vocab, 128) < kSlots;
}

// groups that fill the device's slots twice over the row tiles (an even load
// with few partials), at most one per vocabulary tile
int fwd_groups(int64_t rows, int64_t vocab) {
  const int64_t row_tiles = std::max<int64_t>(1, tiles_of(rows, narrow(rows, vocab) ? 64 : 128));
  return (int)std::min<int64_t>(tiles_of(vocab, 128), std::max<int64_t>(16, tiles_of(2 * kSlots, row_tiles)));
}

int fwd(const float* hidden, int64_t ld_h, const float* weight, int64_t ld_w, const int64_t* target, int64_t rows,
        int64_t dim, int64_t vocab, float* logprob, float* entropy, float* lse, float* partial, hipStream_t s) {
  const int groups = fwd_groups(rows, vocab);
  const bool nar = narrow(rows, vocab), vec = vec_ok(hidden, ld_h) && vec_ok(weight, ld_w);
  const int tok_tiles = (int)tiles_of(rows, nar ? 64 : 128);
  {
    ts::TimedLaunch timed_("logprob.f32_fwd_stats_kernel", s);
    auto run = [&](auto kernel) {
      hipLaunchKernelGGL(kernel, dim3((unsigned)(tok_tiles * groups)), dim3(kThreads), 0, s, hidden, ld_h, weight,
                         ld_w, rows, dim, vocab, groups, tok_tiles, partial);
    };
    if (nar) vec ? run(fwd_stats_kernel<1, true>) : run(fwd_stats_kernel<1, false>);
    else vec ? run(fwd_stats_kernel<2, true>) : run(fwd_stats_kernel<2, false>);
  }
  {
    ts::TimedLaunch timed_("logprob.f32_combine_kernel", s);
    hipLaunchKernelGGL(combine_kernel, dim3((unsigned)((rows + 3) / 4)), dim3(kThreads), 0, s, partial, groups, hidden,
                       ld_h, weight, ld_w, target, rows, dim, vocab, logprob, entropy, lse);
  }
  return ts::check_launch("ts_logprob_fwd_exact");
}

int dlogits(const float* hidden, int64_t ld_h, const float* weight, int64_t ld_w, const int64_t* target,
            const float* lse, const float* ent, const float* g_lp, const float* g_ent, int64_t rows, int64_t dim,
            int64_t vocab, float* dl, int64_t ld_dl, hipStream_t s) {
  const bool nar = narrow(rows, vocab), vec = vec_ok(hidden, ld_h) && vec_ok(weight, ld_w);
  const int tok_tiles = (int)tiles_of(rows, nar ? 64 : 128), v_tiles = (int)tiles_of(vocab, 128);
  ts::TimedLaunch timed_("logprob.f32_dlogits_kernel", s);
  auto run = [&](auto kernel) {
    hipLaunchKernelGGL(kernel, dim3((unsigned)(tok_tiles * v_tiles)), dim3(kThreads), 0, s, hidden, ld_h, weight, ld_w,
                       target, lse, ent, g_lp, g_ent, rows, dim, vocab, dl, ld_dl, tok_tiles, v_tiles);
  };
  if (nar) vec ? run(dlogits_kernel<1, true>) : run(dlogits_kernel<1, false>);
  else vec ? run(dlogits_kernel<2, true>) : run(dlogits_kernel<2, false>);
  return ts::check_launch("ts_logprob_dlogits_exact");
}

// contraction ranges: as many as fill the device's slots once when the tiles
// alone leave some empty, each at least 512 long and of whole stages
void matmul_split(int64_t m, int64_t n, int64_t k, int& mi, int& ranges, int64_t& kper) {
  mi = m <= 64 ? 1 : 2;
  const int64_t tiles = tiles_of(m, 64 * mi) * tiles_of(n, 128);
  int64_t r = tiles > 0 ? kSlots / tiles : 1;
  r = std::max<int64_t>(1, std::min<int64_t>(r, k / 512));
  kper = std::max<int64_t>(BKF, tiles_of(tiles_of(k, r), BKF) * BKF);
  ranges = (int)std::max<int64_t>(1, tiles_of(k, kper));
}

int64_t matmul_workspace(int64_t m, int64_t n, int64_t k) {
  int mi, ranges;
  int64_t kper;
  matmul_split(m, n, k, mi, ranges, kper);
  return ranges > 1 ? ranges * m * n * (int64_t)sizeof(float) : 0;
}

template <int MI, bool KFA, bool KFB>
void launch_matmul(bool vec, unsigned grid, hipStream_t s, const float* a, int64_t a_m, int64_t a_k, const float* b,
                   int64_t b_k, int64_t b_n, int64_t m, int64_t n, int64_t k, float* c, int64_t ldc, int accumulate,
                   int m_tiles, int n_tiles, int ranges, int64_t kper, float* part) {
  auto run = [&](auto kernel) {
    hipLaunchKernelGGL(kernel, dim3(grid), dim3(kThreads), 0, s, a, a_m, a_k, b, b_k, b_n, m, n, k, c, ldc, accumulate,
                       m_tiles, n_tiles, ranges, kper, part);
  };
  vec ? run(matmul_kernel<MI, KFA, KFB, true>) : run(matmul_kernel<MI, KFA, KFB, false>);
}

int matmul(const float* a, int64_t a_m, int64_t a_k, const float* b, int64_t b_k, int64_t b_n, int64_t m, int64_t n,
           int64_t k, float* c, int64_t ldc, int accumulate, float* part, hipStream_t s) {
  int mi, ranges;
  int64_t kper;
  matmul_split(m, n, k, mi, ranges, kper);
  if (!part) {
    ranges = 1;
    kper = std::max<int64_t>(k, 1);
  }
  const int m_tiles = (int)tiles_of(m, 64 * mi), n_tiles = (int)tiles_of(n, 128);
  const bool kfa = a_k == 1, kfb = b_k == 1;
  // 16-byte loads run along the unit-stride index of each operand
  const bool vec = (kfa ? vec_ok(a, a_m) : a_m == 1 && vec_ok(a, a_k)) &&
                   (kfb ? vec_ok(b, b_n) : b_n == 1 && vec_ok(b, b_k));
  const unsigned grid = (unsigned)((int64_t)m_tiles * n_tiles * ranges);
  {
    ts::TimedLaunch timed_("logprob.f32_matmul_kernel", s);
#define LPF_MATMUL(MI, KFA, KFB)                                                                                  \
  launch_matmul<MI, KFA, KFB>(vec, grid, s, a, a_m, a_k, b, b_k, b_n, m, n, k, c, ldc, accumulate, m_tiles,      \
                              n_tiles, ranges, kper, part)
    if (mi == 1) {
      if (kfa) kfb ? LPF_MATMUL(1, true, true) : LPF_MATMUL(1, true, false);
      else kfb ? LPF_MATMUL(1, false, true) : LPF_MATMUL(1, false, false);
    } else {
      if (kfa) kfb ? LPF_MATMUL(2, true, true) : LPF_MATMUL(2, true, false);
      else kfb ? LPF_MATMUL(2, false, true) : LPF_MATMUL(2, false, false);
    }
#undef LPF_MATMUL
  }
  int st = ts::check_launch("ts_matmul_exact");
  if (st != TS_OK || ranges == 1) return st;
  {
    ts::TimedLaunch timed_("logprob.f32_reduce_kernel", s);
    hipLaunchKernelGGL(reduce_kernel, dim3((unsigned)tiles_of(m * n, kThreads)), dim3(kThreads), 0, s, part, ranges, m,
                       n, c, ldc, accumulate);
  }
  return ts::check_launch("ts_matmul_exact (reduce)");
}

}  // namespace lpf
}  // namespace ts
