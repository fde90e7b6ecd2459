// Chunked-vocab fused log-probability / entropy and its gradient with respect
// to the hidden states, for gfx950 (bf16 operands, fp32 accumulation).
//
// Reference: accel/fused_logprob.py:61-338.  The reference materialises one
// fp32 [chunk, V] logit block per chunk and makes several passes over it; here
// the logits never leave the MFMA accumulators:
//
//   forward   logits^T tile = W_tile . H_tile^T on MFMA (A = vocab rows of W,
//             B = token rows of H, both K-contiguous).  The epilogue reduces
//             each token column of the tile to (max, sum exp, sum exp*(l-max));
//             a combine kernel merges the per-tile partials into logprob,
//             entropy and lse and takes the target logit as a dot product.  HBM traffic: W once,
//             H once per vocab super-tile, partials (12 bytes/token/tile).
//   backward  the same tile GEMM recomputes the logits; the epilogue forms
//             dlogits = -p (g_lp + g_H (log p + H)) + g_lp [v == t] in
//             registers, rounds it to bf16 (the reference rounds dlogits to the
//             hidden dtype before its VJP GEMM, fused_logprob.py:165, :295) and
//             stores a [rows, V] bf16 block; a second GEMM multiplies it by
//             W, read in place (its rows are the contraction index), into dh,
//             and for a trainable head a third by the hidden states into dW.
//
// GEMM core (gemm_core.h): work-group tiles of 256 vocabulary rows (or hidden
// dims) x 64 to 320 tokens on v_mfma_f32_32x32x16_bf16, K streamed through a
// 4-stage LDS ring by buffer_load ... lds.
#include <algorithm>
#include <type_traits>

#include "common.h"
#include "gemm_core.h"
#include "timing.h"
#include "../../include/thundersync_hip.h"

namespace ts {
namespace lp {

using namespace ts::gemm;

constexpr int kThreads = 256;      // grad_hidden_reduce_kernel
constexpr int BM = TM;   // vocab rows per forward partial
constexpr float kLog2e = 1.4426950408889634f;
constexpr float kLn2 = 0.6931471805599453f;
__device__ __forceinline__ float neg_inf() { return -__builtin_huge_valf(); }

// (max, sum exp(l - max), sum exp(l - max) (l - max)) of two disjoint sets of
// logits, either of which may be empty (max = -inf, sums 0).  A set of logits of
// -inf counts as empty; the sums of one that holds a NaN, which no maximum shows,
// are NaN.
__device__ __forceinline__ void merge_stats(float& m, float& s, float& e, float mo, float so, float eo) {
  if (mo == neg_inf() || m == neg_inf()) {
    m = fmaxf(m, mo);
    s += so;
    e += eo;
    return;
  }
  const float mn = fmaxf(m, mo);
  const float a = fast_exp2((m - mn) * kLog2e);
  const float b = fast_exp2((mo - mn) * kLog2e);
  e = a * (e + s * (m - mn)) + b * (eo + so * (mo - mn));
  s = a * s + b * so;
  m = mn;
}

// ---------------------------------------------------------------------------
// forward: per (vocab tile, token tile) partial softmax statistics
// ---------------------------------------------------------------------------
struct FwdArgs {
  const bf16* h;
  int64_t ldh;
  const bf16* w;
  int64_t ldw;
  int rows, dim, vocab;
  int n_ttiles, n_vtiles;
  float* part_m;   // [n_vtiles][rows]
  float* part_s;
  float* part_e;
};

// Token rows per tile of a launch: the rows spread evenly over as few tiles as
// 256-token tiles take.  Rows past the end of a tile are MFMA work on zeros --
// cheap on a chip whose clock follows its power, so a narrower tile pays only
// where it is much narrower: 64 or 128 tokens (4096 x 151936: 25 rows forward 279
// -> 264, dlogits 307 -> 269, grad_hidden 201 -> 188 us, 128 rows 307 -> 288, 337 ->
// 295, 235 -> 223), and for grad_hidden, whose launch of few rows is one round that
// ends with its widest tiles, 192 for up to 160 (320 rows 463 -> 409; at 192 rows a
// tile 464 -> 478, and forward and dlogits gain nothing).
inline int token_tile(int64_t rows, bool up_to_192) {
  const int64_t tiles = (rows + TN - 1) / TN, each = (rows + tiles - 1) / tiles;
  return each <= 64 ? 64 : each <= 128 ? 128 : up_to_192 && each <= 160 ? 192 : 256;
}

// The 320-token tile (Wide) reads a weight tile once for rows that need two or
// more 256-token ones, in kWideCost / 256 of a 256-token tile's time (by its MFMAs
// 320 / 256; set to what the launches below take).  `stride`: the token
// operand's, for the 32-bit offsets of its rows within a tile.
constexpr int kWideTokens = Wide::BN;
constexpr int kWideCost = 352;
inline bool wide_fits(int64_t rows, int64_t stride) { return rows > TN && (kWideTokens - 1) * stride < (1ll << 30); }

// Forward and dlogits: 320 where the launch then takes less time in rounds of one
// work-group per CU: 1 tile for 2 at 257 .. 320 rows of 594 vocabulary tiles (3
// rounds for 5: 281 rows forward 488 -> 434 us, dlogits 500 -> 450), 2 for 3 at 600 (5
// for 7: 755 -> 698, 778 -> 723), but not at 384 (5 for 5: 520 -> 651) or 2048 (17 for
// 19: 2157 -> 2286).
inline int logits_tile(int64_t rows, int64_t vtiles, int64_t stride) {
  auto rounds = [&](int64_t w) { return ((rows + w - 1) / w * vtiles + 255) / 256; };
  if (wide_fits(rows, stride) && rounds(kWideTokens) * kWideCost < rounds(TN) * TN) return kWideTokens;
  return token_tile(rows, false);
}

template <typename E, class S>
__global__ __launch_bounds__(kGemmThreads, 1) void fwd_stats_kernel(FwdArgs p) {
  GEMM_RING_OF(S)
  constexpr int MI = S::MI, NI = S::NI;
  const int total = p.n_ttiles * p.n_vtiles;
  int vt, tt;
  grouped_tile(xcd_logical(blockIdx.x, total), p.n_vtiles, p.n_ttiles, vt, tt);
  const int v0 = vt * TM, n0 = tt * S::BN;
  f32x16 acc[MI][NI];
  gemm_tile<E, false, false, S>(acc, p.w + (int64_t)v0 * p.ldw, p.ldw, min(TM, p.vocab - v0),
                          p.h + (int64_t)n0 * p.ldh, p.ldh, min(S::BN, p.rows - n0), p.dim, s0, s1, s2, s3);
  const int tid = threadIdx.x, lane = tid & 63, wave = tid >> 6;
  const int wm = wave % S::WM, wn = wave / S::WM;
  float* xm = reinterpret_cast<float*>(s0);  // [WM - 1][BN] per token, from the waves wm > 0
  float* xs = xm + (S::WM - 1) * S::BN;
  float* xe = xs + (S::WM - 1) * S::BN;
  // rows past the vocabulary (last vocab tile only) take no part
  if (v0 + TM > p.vocab) {
#pragma unroll
    for (int mi = 0; mi < MI; ++mi)
#pragma unroll
      for (int ni = 0; ni < NI; ++ni)
#pragma unroll
        for (int i = 0; i < 16; ++i)
          if (v0 + a_row<S>(mi, i, lane, wm) >= p.vocab) acc[mi][ni][i] = neg_inf();
  }
  float mk[NI], sk[NI], ek[NI];  // this lane's column statistics, kept across the exchange
#pragma unroll
  for (int ni = 0; ni < NI; ++ni) {
    const int col = b_row<S>(ni, lane, wn);
    float m = neg_inf();
#pragma unroll
    for (int mi = 0; mi < MI; ++mi)
#pragma unroll
      for (int i = 0; i < 16; i += 2) m = fmaxf(m, fmaxf(acc[mi][ni][i], acc[mi][ni][i + 1]));
    // sum of q = 2^d2 and of q d2 with d2 = (l - m) log2 e as one FMA per logit; the second
    // sum is taken back to natural-log units once
    float sum = 0.f, e = 0.f;
    const float m2 = m * kLog2e;
    if (m == neg_inf()) {
#pragma unroll
      for (int mi = 0; mi < MI; ++mi)
#pragma unroll
        for (int i = 0; i < 16; ++i)
          if (acc[mi][ni][i] != neg_inf()) sum = e = __builtin_nanf("");
    } else if (v0 + TM <= p.vocab) {
#pragma unroll
      for (int mi = 0; mi < MI; ++mi)
#pragma unroll
        for (int i = 0; i < 16; ++i) {
          const float d2 = fmaf(acc[mi][ni][i], kLog2e, -m2);
          const float q = fast_exp2(d2);
          sum += q;
          e = fmaf(q, d2, e);
        }
    } else {
#pragma unroll
      for (int mi = 0; mi < MI; ++mi)
#pragma unroll
        for (int i = 0; i < 16; ++i) {
          const float d2 = fmaf(acc[mi][ni][i], kLog2e, -m2);  // -inf past the vocabulary: q = 0
          const float q = fast_exp2(d2);
          sum += q;
          e = q > 0.f ? fmaf(q, d2, e) : e;
        }
    }
    e *= kLn2;
    // merge with the other half-wave (lane ^ 32 holds the other vocab rows)
    {
      const float mo = shfl_xor(m, 32), so = shfl_xor(sum, 32), eo = shfl_xor(e, 32);
      merge_stats(m, sum, e, mo, so, eo);
    }
    if (wm > 0 && lane < 32) {
      xm[(wm - 1) * S::BN + col] = m;
      xs[(wm - 1) * S::BN + col] = sum;
      xe[(wm - 1) * S::BN + col] = e;
    }
    mk[ni] = m;
    sk[ni] = sum;
    ek[ni] = e;
  }
  __syncthreads();  // one exchange for both column groups (their columns differ)
#pragma unroll
  for (int ni = 0; ni < NI; ++ni) {
    const int col = b_row<S>(ni, lane, wn);
    const int n = n0 + col;
    if (wm == 0 && lane < 32 && n < p.rows) {
#pragma unroll
      for (int w = 0; w < S::WM - 1; ++w)
        merge_stats(mk[ni], sk[ni], ek[ni], xm[w * S::BN + col], xs[w * S::BN + col], xe[w * S::BN + col]);
      const int64_t o = (int64_t)vt * p.rows + n;
      p.part_m[o] = mk[ni];
      p.part_s[o] = sk[ni];
      p.part_e[o] = ek[ni];
    }
  }
}

// Merge the per-vocab-tile partials of each token and form its target logit
// l[n, t] = sum_d h[n, d] W[t, d] (fp32 sum of exact 16-bit products; NaN logprob
// for t outside [0, vocab)).  A work-group of 16 waves owns 16 tokens: its 64
// slots of 16 lanes merge the tiles t = slot, slot + 64, ... (a slot reads 64
// consecutive bytes of one tile's row of partials), then the 4 slots of a wave
// and the 16 waves meet in a fixed order, while wave w takes token w's dot
// product.  Bound by the latency of the tile loop, so the tiles are cut over as
// many slots as a work-group holds and the rows over 16-token work-groups: 64
// tokens per four-wave work-group walked 149 tiles one after another (400 rows of
// 594 tiles: 131 us and a target-logit launch of 7 us, now 21 us).
constexpr int kCombineTokens = 16;
constexpr int kCombineThreads = 64 * kCombineTokens;

template <typename E>
__global__ __launch_bounds__(kCombineThreads) void combine_kernel(
    const float* __restrict__ pm, const float* __restrict__ ps, const float* __restrict__ pe,
    const bf16* __restrict__ h, int64_t ldh, const bf16* __restrict__ w, int64_t ldw,
    const int64_t* __restrict__ target, int rows, int dim, int n_vtiles, int vocab, float* __restrict__ logprob,
    float* __restrict__ entropy, float* __restrict__ lse) {
  __shared__ float sm[16][16], ss[16][16], se[16][16], st[16];
  const int lane = threadIdx.x & 63, wave = threadIdx.x >> 6;
  const int tok = lane & 15, slot = 4 * wave + (lane >> 4);
  const int n0 = blockIdx.x * kCombineTokens, n = n0 + tok;
  float M = neg_inf(), S = 0.f, X = 0.f;  // X: sum exp(l - M) (l - M)
  if (n < rows) {
#pragma unroll 4
    for (int t = slot; t < n_vtiles; t += 64) {
      const int64_t o = (int64_t)t * rows + n;
      merge_stats(M, S, X, pm[o], ps[o], pe[o]);
    }
  }
#pragma unroll
  for (int o = 16; o < 64; o <<= 1) {
    const float mo = shfl_xor(M, o), so = shfl_xor(S, o), xo = shfl_xor(X, o);
    merge_stats(M, S, X, mo, so, xo);
  }
  if (lane < 16) {
    sm[wave][tok] = M;
    ss[wave][tok] = S;
    se[wave][tok] = X;
  }
  // wave w: the target logit of token n0 + w
  if (n0 + wave < rows) {
    const int64_t t = target[n0 + wave];
    if (t >= 0 && t < vocab) {
      const bf16* hr = h + (int64_t)(n0 + wave) * ldh;
      const bf16* wr = w + t * ldw;
      float acc = 0.f;
      for (int d = 8 * lane; d < dim; d += 512) {
        const u32x4 a = ld16(hr + d), b = ld16(wr + d);
#pragma unroll
        for (int i = 0; i < 4; ++i) {
          acc = fmaf(bits_to_f<E>(a[i] & 0xffffu), bits_to_f<E>(b[i] & 0xffffu), acc);
          acc = fmaf(bits_to_f<E>(a[i] >> 16), bits_to_f<E>(b[i] >> 16), acc);
        }
      }
      acc = wave_sum(acc);
      if (lane == 0) st[wave] = acc;
    } else if (lane == 0) {
      st[wave] = __builtin_nanf("");
    }
  }
  __syncthreads();
  if (threadIdx.x >= 16 || n >= rows) return;
  M = sm[0][tok];
  S = ss[0][tok];
  X = se[0][tok];
#pragma unroll
  for (int v = 1; v < 16; ++v) merge_stats(M, S, X, sm[v][tok], ss[v][tok], se[v][tok]);
  const float logs = logf(S);
  logprob[n] = (st[tok] - M) - logs;
  lse[n] = M + logs;
  if (entropy) entropy[n] = logs - X / S;
}

// ---------------------------------------------------------------------------
// backward 1: recompute logits, form bf16 dlogits [rows, ld] (pad columns 0)
// ---------------------------------------------------------------------------
struct DlArgs {
  const bf16* h;
  int64_t ldh;
  const bf16* w;
  int64_t ldw;
  const int64_t* target;
  const float* lse;
  const float* ent;
  const float* g_lp;
  const float* g_ent;  // may be null
  int rows, dim, vocab, vocab_pad;
  int n_ttiles, n_vtiles;
  bf16* dl;
  int64_t ldl;
};

constexpr int OPITCH = TM + 8;  // staging pitch (bf16) of [64 tokens][TM vocab] quarter tiles
static_assert(64 * OPITCH <= kRingElems, "a quarter of the dlogits tile fits one ring stage");

// A target lies in one vocabulary tile of 594, so the one-hot term sits behind a
// wave-wide test of whether any of the wave's tokens has its target among the
// wave's rows: compared in every element it also spilled 243 scalar registers of
// comparison masks (dlogits 2.15 -> 2.06 ms per 2048 rows x 4096 x 151936).
template <typename E, class S>
__global__ __launch_bounds__(kGemmThreads, 1) void dlogits_kernel(DlArgs p) {
  GEMM_RING_OF(S)
  constexpr int MI = S::MI, NI = S::NI;
  const int total = p.n_ttiles * p.n_vtiles;
  int vt, tt;
  grouped_tile(xcd_logical(blockIdx.x, total), p.n_vtiles, p.n_ttiles, vt, tt);
  const int v0 = vt * TM, n0 = tt * S::BN;
  f32x16 acc[MI][NI];
  gemm_tile<E, false, false, S>(acc, p.w + (int64_t)v0 * p.ldw, p.ldw, min(TM, p.vocab - v0),
                          p.h + (int64_t)n0 * p.ldh, p.ldh, min(S::BN, p.rows - n0), p.dim, s0, s1, s2, s3);
  const int tid = threadIdx.x, lane = tid & 63, wave = tid >> 6;
  const int wm = wave % S::WM, wn = wave / S::WM;
  // tokens 64 q .. 64 q + 63 of the tile are staged in ring stage q as [64][OPITCH];
  // a Wide tile does not fit, its waves' two halves of the tokens take turns
  constexpr int PASSES = S::BN > TN ? S::WN : 1, PT = S::BN / PASSES;  // tokens per pass
  static_assert(PT <= 256, "four stages of 64 tokens");
  auto quarter = [&](int q) -> bf16* { return q == 0 ? s0 : q == 1 ? s1 : q == 2 ? s2 : s3; };
  // dl = -p (g_lp + g_H (log p + H)) + g_lp [v = t], with log2 p = l log2 e - lse log2 e as one
  // FMA and the bracket as one FMA in log2 p: A = g_H ln 2, B = g_lp + g_H H per token.  Tiles
  // inside the vocabulary (all but the last) skip the bounds test; columns past the rows take
  // the last row's values and are not stored.
  auto column = [&](int ni, auto full_c, auto hot_c, float lse2, float coef_a, float coef_b, float glp, int hot)
                    __attribute__((always_inline)) {
    constexpr bool FULL = decltype(full_c)::value, HOT = decltype(hot_c)::value;
    const int col = b_row<S>(ni, lane, PASSES > 1 ? 0 : wn);  // token within the pass
    bf16* out = quarter(col >> 6) + (col & 63) * OPITCH;
#pragma unroll
    for (int mi = 0; mi < MI; ++mi)
#pragma unroll
      for (int i4 = 0; i4 < 4; ++i4) {
        float d[4];
#pragma unroll
        for (int j = 0; j < 4; ++j) {
          const int i = 4 * i4 + j;
          const float logp2 = fmaf(acc[mi][ni][i], kLog2e, -lse2);
          d[j] = -fast_exp2(logp2) * fmaf(coef_a, logp2, coef_b);
          if (HOT && a_row<S>(mi, i, lane, wm) == hot) d[j] += glp;
          if (!FULL && v0 + a_row<S>(mi, i, lane, wm) >= p.vocab) d[j] = 0.f;
        }
        // vocab rows a_row(mi, 4 i4 .. 4 i4 + 3) are consecutive: one 8-byte write
        *reinterpret_cast<u32x2*>(out + a_row<S>(mi, 4 * i4, lane, wm)) =
            u32x2{pack2<E>(d[0], d[1]), pack2<E>(d[2], d[3])};
      }
  };
  auto epilogue = [&](auto full_c) __attribute__((always_inline)) {
#pragma unroll
    for (int ni = 0; ni < NI; ++ni) {
      const int n = min(n0 + b_row<S>(ni, lane, wn), p.rows - 1);
      const float lse2 = p.lse[n] * kLog2e, glp = p.g_lp[n];
      float coef_a = 0.f, coef_b = glp;
      if (p.g_ent) {
        const float gent = p.g_ent[n];
        coef_a = gent * kLn2;
        coef_b = fmaf(gent, p.ent[n], glp);
      }
      const int64_t t = p.target[n];
      // the token's target as a row of the tile (out-of-range targets match none)
      const int hot = t >= v0 && t < min(v0 + TM, p.vocab) ? (int)(t - v0) : -1;
      const int mine = hot - 32 * MI * wm;
      if (__builtin_amdgcn_ballot_w64(mine >= 0 && mine < 32 * MI) != 0)
        column(ni, full_c, std::true_type{}, lse2, coef_a, coef_b, glp, hot);
      else
        column(ni, full_c, std::false_type{}, lse2, coef_a, coef_b, glp, hot);
      if constexpr (PASSES > 1) __builtin_amdgcn_sched_barrier(0);
    }
  };
  const int vmax = min(TM, p.vocab_pad - v0);
  // coalesced store of the pass's [PT tokens][TM vocab]
  auto store = [&](int pass) __attribute__((always_inline)) {
#pragma unroll 4
    for (int it = 0; it < (PT * TM / 8) / kGemmThreads; ++it) {
      const int c = it * kGemmThreads + tid;
      const int row = c / (TM / 8), chunk = (c % (TM / 8)) * 8;
      const int n = n0 + pass * PT + row;
      if (n < p.rows && chunk < vmax)
        *reinterpret_cast<u32x4*>(p.dl + (int64_t)n * p.ldl + v0 + chunk) =
            *reinterpret_cast<const u32x4*>(quarter(row >> 6) + (row & 63) * OPITCH + chunk);
    }
  };
  auto values = [&]() __attribute__((always_inline)) {
    if (v0 + TM <= p.vocab) epilogue(std::true_type{});
    else epilogue(std::false_type{});
  };
  if constexpr (PASSES == 1) {
    values();
    __syncthreads();
    store(0);
  } else {
    static_assert(PASSES <= 2, "two halves");
    if (wn == 0) values();
    __syncthreads();
    store(0);
    __syncthreads();
    if (wn == 1) values();
    __syncthreads();
    store(1);
  }
}

// ---------------------------------------------------------------------------
// backward 2: grad_hidden[n][d] = sum_v dl[n][v] W[v][d] as C^T = W^T . dl^T,
// W read in place as a K-strided operand (its rows are the contraction
// index).  With `ksplit` > 1 the vocabulary is cut into ksplit ranges of
// whole stages; range s of every tile writes fp32 partial sums to
// part[s][n][d] and grad_hidden_reduce_kernel adds them in range order.
// ---------------------------------------------------------------------------
struct DhArgs {
  const bf16* w;    // [vocab][ldw]
  int64_t ldw;
  const bf16* dl;   // [rows][ldl]
  int64_t ldl;
  int rows, dim, vocab;
  int n_ttiles, n_dtiles, ksplit, kper;  // kper: vocabulary per range (multiple of TK)
  bf16* dh;
  int64_t ldd;
  float* part;      // [ksplit][rows][dim] when ksplit > 1
};

template <typename E, class S>
__global__ __launch_bounds__(kGemmThreads, 1) void grad_hidden_kernel(DhArgs p) {
  GEMM_RING_OF(S)
  constexpr int MI = S::MI, NI = S::NI;
  const int tiles = p.n_ttiles * p.n_dtiles;
  const int id = xcd_logical(blockIdx.x, tiles * p.ksplit);
  const int ks = id / tiles;  // vocabulary range: tiles of one range run together
  int dt, tt;
  grouped_tile(id - ks * tiles, p.n_dtiles, p.n_ttiles, dt, tt);
  const int d0 = dt * TM, n0 = tt * S::BN;
  const int kb = ks * p.kper, ke = min(p.vocab, kb + p.kper);
  f32x16 acc[MI][NI];
  gemm_tile<E, true, false, S>(acc, p.w + (int64_t)kb * p.ldw + d0, p.ldw, p.dim - d0,
                               p.dl + (int64_t)n0 * p.ldl + kb, p.ldl, min(S::BN, p.rows - n0), ke - kb, s0, s1, s2,
                               s3);
  const int lane = threadIdx.x & 63, wave = threadIdx.x >> 6;
  const int wm = wave % S::WM, wn = wave / S::WM;
#pragma unroll
  for (int ni = 0; ni < NI; ++ni) {
    const int n = n0 + b_row<S>(ni, lane, wn);
    if (n >= p.rows) continue;
#pragma unroll
    for (int mi = 0; mi < MI; ++mi)
#pragma unroll
      for (int i4 = 0; i4 < 4; ++i4) {
        const int d = d0 + a_row<S>(mi, 4 * i4, lane, wm);
        const float a[4] = {acc[mi][ni][4 * i4], acc[mi][ni][4 * i4 + 1], acc[mi][ni][4 * i4 + 2],
                            acc[mi][ni][4 * i4 + 3]};
        if (p.ksplit > 1) {
          float* q = p.part + ((int64_t)ks * p.rows + n) * p.dim + d;
          if (d + 3 < p.dim) {
            *reinterpret_cast<f32x4*>(q) = f32x4{a[0], a[1], a[2], a[3]};
          } else {
            for (int j = 0; j < 4; ++j)
              if (d + j < p.dim) q[j] = a[j];
          }
        } else if (d + 3 < p.dim) {
          *reinterpret_cast<u32x2*>(p.dh + (int64_t)n * p.ldd + d) = u32x2{pack2<E>(a[0], a[1]), pack2<E>(a[2], a[3])};
        } else {
          for (int j = 0; j < 4; ++j)
            if (d + j < p.dim) reinterpret_cast<E*>(p.dh)[(int64_t)n * p.ldd + d + j] = from_f<E>(a[j]);
        }
      }
  }
}

// dh = bf16(sum_s part[s]) in range order; four elements per thread
template <typename E>
__global__ __launch_bounds__(kThreads) void grad_hidden_reduce_kernel(const float* __restrict__ part, int ksplit,
                                                                      int rows, int dim, bf16* __restrict__ dh,
                                                                      int64_t ldd) {
  const int64_t e = ((int64_t)blockIdx.x * kThreads + threadIdx.x) * 4;
  const int64_t total = (int64_t)rows * dim;
  if (e >= total) return;
  const int64_t n = e / dim;
  const int d = (int)(e - n * dim);
  f32x4 s = *reinterpret_cast<const f32x4*>(part + e);
  for (int k = 1; k < ksplit; ++k) s += *reinterpret_cast<const f32x4*>(part + (int64_t)k * total + e);
  *reinterpret_cast<u32x2*>(dh + n * ldd + d) = u32x2{pack2<E>(s[0], s[1]), pack2<E>(s[2], s[3])};
}

// ---------------------------------------------------------------------------
// backward 3 (trainable head): grad_weight[v][d] = sum_n dl[n][v] h[n][d] as
// C = dl^T . h with both operands K-strided (K = the block's rows), in fp32
// over the blocks in block order.  The first block writes the fp32
// accumulator without reading it and the last one adds it to its tile and
// writes the gradient in the element type, so a gradient of one block needs
// no accumulator and one of two blocks one write and one read of it, with no
// zero fill before and no cast pass after.  A tile's epilogue is bound by the
// accumulator's latency (nothing else runs on the CU meanwhile): it takes 16
// accumulator values at a time, all loads before the first store.  4096 rows x
// 2048 x 151936 in two blocks: 4.42 ms, a 0.16 ms fill and a 0.30 ms cast with
// one read-add-write per value, 2.57 ms in all now (0.99 PFLOP/s).
// ---------------------------------------------------------------------------
struct DwArgs {
  const bf16* dl;   // [rows][ldl]
  int64_t ldl;
  const bf16* h;    // [rows][ldh]
  int64_t ldh;
  int rows, dim, vocab;
  int n_vtiles, n_dtiles;
  const float* gw_in;  // [vocab][ldg] the earlier blocks' sum, or null
  float* gw;           // [vocab][ldg] the sum with this block, or null:
  int64_t ldg;
  bf16* out;           // [vocab][ldo] rounded to the element type
  int64_t ldo;
};

template <typename E>
__global__ __launch_bounds__(kGemmThreads, 1) void grad_weight_kernel(DwArgs p) {
  GEMM_RING
  const int total = p.n_vtiles * p.n_dtiles;
  int vt, dt;
  grouped_tile(xcd_logical(blockIdx.x, total), p.n_vtiles, p.n_dtiles, vt, dt);
  const int v0 = vt * TM, d0 = dt * TN;
  f32x16 acc[4][NI];
  gemm_tile<E, true, true>(acc, p.dl + v0, p.ldl, p.vocab - v0, p.h + d0, p.ldh, p.dim - d0, p.rows, s0, s1, s2,
                        s3);
  const int lane = threadIdx.x & 63, wave = threadIdx.x >> 6;
  const int wm = wave & 1, wn = wave >> 1;
#pragma unroll
  for (int ni = 0; ni < NI; ++ni) {
    const int d = d0 + b_row(ni, lane, wn);
    if (d >= p.dim) continue;
#pragma unroll
    for (int mi = 0; mi < 4; ++mi) {
      // rows past the vocabulary read its last row and store nothing
      if (p.gw_in) {
        float g[16];
#pragma unroll
        for (int i = 0; i < 16; ++i)
          g[i] = p.gw_in[(int64_t)min(v0 + a_row(mi, i, lane, wm), p.vocab - 1) * p.ldg + d];
#pragma unroll
        for (int i = 0; i < 16; ++i) acc[mi][ni][i] += g[i];
      }
#pragma unroll
      for (int i = 0; i < 16; ++i) {
        const int v = v0 + a_row(mi, i, lane, wm);
        if (v >= p.vocab) continue;
        if (p.gw) p.gw[(int64_t)v * p.ldg + d] = acc[mi][ni][i];
        else reinterpret_cast<E*>(p.out)[(int64_t)v * p.ldo + d] = from_f<E>(acc[mi][ni][i]);
      }
    }
  }
}

// ksplit (vocabulary ranges) for grad_hidden: as many ranges as keep the
// launch within one round of 256 work-groups (one per CU) when the row tiles
// alone do not fill it -- a second, partial round would cost a whole range's
// time (80 tiles: three ranges of a third, not four of a quarter in two
// rounds) -- each range at least 4096 vocabulary rows.  `width`: token rows per
// tile, 320 where the launch of its tiles and ranges takes less time
// (4096 x 151936: 281 rows 437 -> 351 us, 600 728 -> 618).  Returns the number of token tiles.
inline int grad_hidden_split(int64_t rows, int64_t dim, int64_t vocab, int64_t stride, int& width, int& ksplit,
                             int& kper) {
  const int64_t dtiles = (dim + TM - 1) / TM;
  auto ranges = [&](int64_t w) {
    int64_t k = 256 / ((rows + w - 1) / w * dtiles);
    k = std::min<int64_t>(k, std::max<int64_t>(1, vocab / 4096));
    return std::max<int64_t>(1, std::min<int64_t>(k, 16));
  };
  // time of a launch: rounds x tile width / ranges
  auto time = [&](int64_t w, int cost) {
    const int64_t k = ranges(w), groups = (rows + w - 1) / w * dtiles * k;
    return (double)((groups + 255) / 256 * cost) / (double)k;
  };
  width = token_tile(rows, true);
  if (wide_fits(rows, stride) && time(kWideTokens, kWideCost) < time(width, width)) width = kWideTokens;
  const int64_t k = ranges(width);
  int64_t per = (vocab + k - 1) / k;
  per = (per + TK - 1) / TK * TK;
  ksplit = (int)((vocab + per - 1) / per);
  kper = (int)per;
  return (int)((rows + width - 1) / width);
}

// launch kernel<element, tile shape> by a DType code and token_tile's width
#define TS_LAUNCH_TOKENS(dtype, width, kernel, ...)                               \
  do {                                                                            \
    if ((width) == 64) TS_LAUNCH_E_T(dtype, kernel, Narrow<1>, __VA_ARGS__);      \
    else if ((width) == 128) TS_LAUNCH_E_T(dtype, kernel, Narrow<2>, __VA_ARGS__); \
    else if ((width) == kWideTokens) TS_LAUNCH_E_T(dtype, kernel, Wide, __VA_ARGS__); \
    else TS_LAUNCH_E_T(dtype, kernel, Full, __VA_ARGS__);                         \
  } while (0)

bool ok16(const void* p) { return ((uintptr_t)p & 15) == 0; }

}  // namespace lp
}  // namespace ts

extern "C" {

int64_t ts_logprob_fwd_workspace(int64_t rows, int64_t vocab) {
  if (rows <= 0 || vocab <= 0) return 0;
  const int64_t vt = (vocab + ts::lp::BM - 1) / ts::lp::BM;
  return 3 * vt * rows * (int64_t)sizeof(float);
}

int ts_logprob_fwd(const void* hidden, int64_t ld_hidden, const void* weight, int64_t ld_weight,
                   const int64_t* target, int64_t rows, int64_t dim, int64_t vocab, float* logprob,
                   float* entropy, float* lse, void* workspace, int64_t workspace_bytes, int dtype,
                   void* stream) {
  using namespace ts::lp;
  TS_CHECK_ARG(dtype == ts::kBF16 || dtype == ts::kF16, "ts_logprob_fwd: dtype %d (bf16 or fp16)", dtype);
  TS_CHECK_ARG(rows >= 0 && dim > 0 && vocab > 0 && rows < (1 << 30) && vocab < (1 << 30) &&
                   dim < (1 << 20),
               "ts_logprob_fwd: bad shape rows=%lld dim=%lld vocab=%lld", (long long)rows,
               (long long)dim, (long long)vocab);
  if (rows == 0) return TS_OK;
  TS_CHECK_ARG(hidden && weight && target && logprob && lse, "ts_logprob_fwd: null pointer");
  TS_CHECK_ARG(dim % 8 == 0 && ld_hidden % 8 == 0 && ld_weight % 8 == 0 && ld_hidden >= dim &&
                   ld_weight >= dim && ok16(hidden) && ok16(weight),
               "ts_logprob_fwd: hidden/weight rows must be 16-byte aligned with dim %% 8 == 0");
  TS_CHECK_ARG(255 * ld_hidden < (1ll << 30) && 255 * ld_weight < (1ll << 30),
               "ts_logprob_fwd: leading dimensions too large for 32-bit tile offsets");
  TS_CHECK_ARG(workspace && workspace_bytes >= ts_logprob_fwd_workspace(rows, vocab),
               "ts_logprob_fwd: workspace of %lld bytes, need %lld", (long long)workspace_bytes,
               (long long)ts_logprob_fwd_workspace(rows, vocab));
  FwdArgs a;
  a.h = (const ts::bf16*)hidden;
  a.ldh = ld_hidden;
  a.w = (const ts::bf16*)weight;
  a.ldw = ld_weight;
  a.rows = (int)rows;
  a.dim = (int)dim;
  a.vocab = (int)vocab;
  a.n_vtiles = (int)((vocab + BM - 1) / BM);
  const int width = logits_tile(rows, a.n_vtiles, ld_hidden);
  a.n_ttiles = (int)((rows + width - 1) / width);
  float* ws = (float*)workspace;
  a.part_m = ws;
  a.part_s = ws + (int64_t)a.n_vtiles * rows;
  a.part_e = ws + 2 * (int64_t)a.n_vtiles * rows;
  TS_CHECK_ARG((int64_t)a.n_ttiles * a.n_vtiles < (1ll << 31), "ts_logprob_fwd: grid too large");
  hipStream_t s = (hipStream_t)stream;
  { ts::TimedLaunch timed_("logprob.fwd_stats_kernel", s); TS_LAUNCH_TOKENS(dtype, width, fwd_stats_kernel, dim3((unsigned)(a.n_ttiles * a.n_vtiles)), dim3(kGemmThreads),
                     0, s, a); }
  int st = ts::check_launch("ts_logprob_fwd (tiles)");
  if (st != TS_OK) return st;
  {
    ts::TimedLaunch timed_("logprob.combine_kernel", s);
    TS_LAUNCH_E(dtype, combine_kernel, dim3((unsigned)((rows + kCombineTokens - 1) / kCombineTokens)),
                dim3(kCombineThreads), 0, s, a.part_m, a.part_s, a.part_e, a.h, a.ldh, a.w, a.ldw, target, (int)rows,
                (int)dim, a.n_vtiles, (int)vocab, logprob, entropy, lse);
  }
  return ts::check_launch("ts_logprob_fwd (combine)");
}

int ts_logprob_dlogits(const void* hidden, int64_t ld_hidden, const void* weight, int64_t ld_weight,
                       const int64_t* target, const float* lse, const float* entropy,
                       const float* grad_lp, const float* grad_ent, int64_t rows, int64_t dim,
                       int64_t vocab, void* dlogits, int64_t ld_dlogits, int dtype, void* stream) {
  using namespace ts::lp;
  TS_CHECK_ARG(dtype == ts::kBF16 || dtype == ts::kF16, "ts_logprob_dlogits: dtype %d (bf16 or fp16)", dtype);
  TS_CHECK_ARG(rows >= 0 && dim > 0 && vocab > 0 && rows < (1 << 30) && vocab < (1 << 30) &&
                   dim < (1 << 20),
               "ts_logprob_dlogits: bad shape");
  if (rows == 0) return TS_OK;
  TS_CHECK_ARG(hidden && weight && target && lse && grad_lp && dlogits,
               "ts_logprob_dlogits: null pointer");
  TS_CHECK_ARG(!grad_ent || entropy, "ts_logprob_dlogits: grad_ent needs the saved entropy");
  TS_CHECK_ARG(dim % 8 == 0 && ld_hidden % 8 == 0 && ld_weight % 8 == 0 && ok16(hidden) &&
                   ok16(weight) && ok16(dlogits) && ld_dlogits % 8 == 0 && ld_dlogits >= vocab,
               "ts_logprob_dlogits: alignment (16 bytes, dims %% 8) or ld_dlogits");
  TS_CHECK_ARG(255 * ld_hidden < (1ll << 30) && 255 * ld_weight < (1ll << 30),
               "ts_logprob_dlogits: leading dimensions too large for 32-bit tile offsets");
  DlArgs a;
  a.h = (const ts::bf16*)hidden;
  a.ldh = ld_hidden;
  a.w = (const ts::bf16*)weight;
  a.ldw = ld_weight;
  a.target = target;
  a.lse = lse;
  a.ent = entropy;
  a.g_lp = grad_lp;
  a.g_ent = grad_ent;
  a.rows = (int)rows;
  a.dim = (int)dim;
  a.vocab = (int)vocab;
  a.vocab_pad = (int)((vocab + 7) / 8 * 8);
  a.n_vtiles = (int)((a.vocab_pad + BM - 1) / BM);
  const int width = logits_tile(rows, a.n_vtiles, ld_hidden);
  a.n_ttiles = (int)((rows + width - 1) / width);
  a.dl = (ts::bf16*)dlogits;
  a.ldl = ld_dlogits;
  TS_CHECK_ARG(a.vocab_pad <= ld_dlogits, "ts_logprob_dlogits: ld_dlogits below padded vocab");
  { ts::TimedLaunch timed_("logprob.dlogits_kernel", (hipStream_t)stream); TS_LAUNCH_TOKENS(dtype, width, dlogits_kernel, dim3((unsigned)(a.n_ttiles * a.n_vtiles)), dim3(kGemmThreads),
                     0, (hipStream_t)stream, a); }
  return ts::check_launch("ts_logprob_dlogits");
}

int64_t ts_logprob_grad_hidden_workspace(int64_t rows, int64_t dim, int64_t vocab) {
  if (rows <= 0 || dim <= 0 || vocab <= 0) return 0;
  int width, ksplit, kper;
  ts::lp::grad_hidden_split(rows, dim, vocab, vocab, width, ksplit, kper);
  return ksplit > 1 ? (int64_t)ksplit * rows * dim * (int64_t)sizeof(float) : 0;
}

}  // extern "C"

namespace ts {

int grad_hidden_launch(const void* dlogits, int64_t ld_dlogits, const void* weight, int64_t ld_weight, int64_t rows,
                       int64_t dim, int64_t vocab, void* grad_hidden, int64_t ld_grad, void* workspace,
                       int64_t workspace_bytes, int dtype, void* stream, const char* label,
                       const char* reduce_label) {
  using namespace ts::lp;
  TS_CHECK_ARG(dtype == ts::kBF16 || dtype == ts::kF16, "ts_logprob_grad_hidden: dtype %d (bf16 or fp16)", dtype);
  TS_CHECK_ARG(rows >= 0 && dim > 0 && vocab > 0 && rows < (1 << 30) && dim < (1 << 20) && vocab < (1 << 30),
               "ts_logprob_grad_hidden: bad shape");
  if (rows == 0) return TS_OK;
  TS_CHECK_ARG(dlogits && weight && grad_hidden && ok16(dlogits) && ok16(weight) && ok16(grad_hidden) &&
                   ld_dlogits % 8 == 0 && ld_weight % 8 == 0 && ld_grad % 8 == 0 && dim % 8 == 0 &&
                   ld_dlogits >= (vocab + 7) / 8 * 8 && ld_weight >= dim && ld_grad >= dim,
               "ts_logprob_grad_hidden: alignment or leading dimensions");
  TS_CHECK_ARG(255 * ld_dlogits < (1ll << 30) && 31 * ld_weight < (1ll << 30),
               "ts_logprob_grad_hidden: leading dimensions too large for 32-bit tile offsets");
  DhArgs a;
  a.w = (const ts::bf16*)weight;
  a.ldw = ld_weight;
  a.dl = (const ts::bf16*)dlogits;
  a.ldl = ld_dlogits;
  a.rows = (int)rows;
  a.dim = (int)dim;
  a.vocab = (int)vocab;
  a.n_dtiles = (int)((dim + TM - 1) / TM);
  int width;
  a.n_ttiles = grad_hidden_split(rows, dim, vocab, ld_dlogits, width, a.ksplit, a.kper);
  a.dh = (ts::bf16*)grad_hidden;
  a.ldd = ld_grad;
  a.part = (float*)workspace;
  if (a.ksplit > 1)
    TS_CHECK_ARG(workspace && workspace_bytes >= ts_logprob_grad_hidden_workspace(rows, dim, vocab) &&
                     ok16(workspace),
                 "ts_logprob_grad_hidden: workspace of %lld bytes, need %lld", (long long)workspace_bytes,
                 (long long)ts_logprob_grad_hidden_workspace(rows, dim, vocab));
  hipStream_t s = (hipStream_t)stream;
  {
    ts::TimedLaunch timed_(label, s);
    const dim3 grid((unsigned)(a.n_ttiles * a.n_dtiles * a.ksplit));
    if (width == 192) TS_LAUNCH_E_T(dtype, grad_hidden_kernel, Narrow<3>, grid, dim3(kGemmThreads), 0, s, a);
    else TS_LAUNCH_TOKENS(dtype, width, grad_hidden_kernel, grid, dim3(kGemmThreads), 0, s, a);
  }
  int st = ts::check_launch("ts_logprob_grad_hidden");
  if (st != TS_OK || a.ksplit == 1) return st;
  const int64_t quads = rows * dim / 4;
  {
    ts::TimedLaunch timed_(reduce_label, s);
    TS_LAUNCH_E(dtype, grad_hidden_reduce_kernel, dim3((unsigned)((quads + kThreads - 1) / kThreads)), dim3(kThreads),
                       0, s, (const float*)workspace, a.ksplit, (int)rows, (int)dim, (ts::bf16*)grad_hidden, ld_grad);
  }
  return ts::check_launch("ts_logprob_grad_hidden (reduce)");
}

}  // namespace ts

extern "C" {

int ts_logprob_grad_hidden(const void* dlogits, int64_t ld_dlogits, const void* weight, int64_t ld_weight,
                           int64_t rows, int64_t dim, int64_t vocab, void* grad_hidden, int64_t ld_grad,
                           void* workspace, int64_t workspace_bytes, int dtype, void* stream) {
  return ts::grad_hidden_launch(dlogits, ld_dlogits, weight, ld_weight, rows, dim, vocab, grad_hidden, ld_grad,
                                workspace, workspace_bytes, dtype, stream, "logprob.grad_hidden_kernel",
                                "logprob.grad_hidden_reduce_kernel");
}

int ts_logprob_grad_weight_block(const void* dlogits, int64_t ld_dlogits, const void* hidden, int64_t ld_hidden,
                                 int64_t rows, int64_t dim, int64_t vocab, float* accumulator,
                                 int64_t ld_accumulator, int first, void* grad_weight, int64_t ld_grad, int dtype,
                                 void* stream) {
  using namespace ts::lp;
  TS_CHECK_ARG(dtype == ts::kBF16 || dtype == ts::kF16, "ts_logprob_grad_weight: dtype %d (bf16 or fp16)", dtype);
  TS_CHECK_ARG(rows >= 0 && dim > 0 && vocab > 0 && rows < (1 << 30) && dim < (1 << 20) && vocab < (1 << 30),
               "ts_logprob_grad_weight: bad shape");
  if (rows == 0 && !first && !grad_weight) return TS_OK;
  TS_CHECK_ARG(rows > 0, "ts_logprob_grad_weight: a first or last block without rows");
  TS_CHECK_ARG(dlogits && hidden && ok16(dlogits) && ok16(hidden) && ld_dlogits % 8 == 0 && ld_hidden % 8 == 0 &&
                   dim % 8 == 0 && ld_dlogits >= vocab && ld_hidden >= dim,
               "ts_logprob_grad_weight: alignment or leading dimensions");
  TS_CHECK_ARG((accumulator || (first && grad_weight)) && (!accumulator || ld_accumulator >= dim) &&
                   (!grad_weight || ld_grad >= dim),
               "ts_logprob_grad_weight: no accumulator, or leading dimensions");
  TS_CHECK_ARG(31 * ld_dlogits < (1ll << 30) && 31 * ld_hidden < (1ll << 30),
               "ts_logprob_grad_weight: leading dimensions too large for 32-bit tile offsets");
  DwArgs a;
  a.dl = (const ts::bf16*)dlogits;
  a.ldl = ld_dlogits;
  a.h = (const ts::bf16*)hidden;
  a.ldh = ld_hidden;
  a.rows = (int)rows;
  a.dim = (int)dim;
  a.vocab = (int)vocab;
  a.n_vtiles = (int)((vocab + TM - 1) / TM);
  a.n_dtiles = (int)((dim + TN - 1) / TN);
  a.gw_in = first ? nullptr : accumulator;
  a.gw = grad_weight ? nullptr : accumulator;
  a.ldg = ld_accumulator;
  a.out = (ts::bf16*)grad_weight;
  a.ldo = ld_grad;
  TS_CHECK_ARG((int64_t)a.n_vtiles * a.n_dtiles < (1ll << 31), "ts_logprob_grad_weight: grid too large");
  {
    ts::TimedLaunch timed_("logprob.grad_weight_kernel", (hipStream_t)stream);
    TS_LAUNCH_E(dtype, grad_weight_kernel, dim3((unsigned)(a.n_vtiles * a.n_dtiles)), dim3(kGemmThreads), 0,
                       (hipStream_t)stream, a);
  }
  return ts::check_launch("ts_logprob_grad_weight");
}

int ts_logprob_grad_weight(const void* dlogits, int64_t ld_dlogits, const void* hidden, int64_t ld_hidden,
                           int64_t rows, int64_t dim, int64_t vocab, float* grad_weight, int64_t ld_grad,
                           int dtype, void* stream) {
  TS_CHECK_ARG(grad_weight || rows == 0, "ts_logprob_grad_weight: null grad_weight");
  return ts_logprob_grad_weight_block(dlogits, ld_dlogits, hidden, ld_hidden, rows, dim, vocab, grad_weight, ld_grad,
                                      0, nullptr, 0, dtype, stream);
}

}  // extern "C"
