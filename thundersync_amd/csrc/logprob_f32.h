// fp32 kernels of the input-precision logprob operators (logprob_f32.hip),
// launched by the C entry points of logprob_exact.hip.
#pragma once

#include "common.h"

namespace ts {
namespace lpf {

// vocabulary groups of the forward: statistics partials per row
int fwd_groups(int64_t rows, int64_t vocab);
int fwd(const float* hidden, int64_t ld_h, const float* weight, int64_t ld_w, const int64_t* target, int64_t rows,
        int64_t dim, int64_t vocab, float* logprob, float* entropy, float* lse, float* partial, hipStream_t s);
int dlogits(const float* hidden, int64_t ld_h, const float* weight, int64_t ld_w, const int64_t* target,
            const float* lse, const float* ent, const float* g_lp, const float* g_ent, int64_t rows, int64_t dim,
            int64_t vocab, float* dl, int64_t ld_dl, hipStream_t s);
// bytes of partial sums matmul wants for its contraction ranges (0: one range)
int64_t matmul_workspace(int64_t m, int64_t n, int64_t k);
// `part` null: one contraction range
int matmul(const float* a, int64_t a_m, int64_t a_k, const float* b, int64_t b_k, int64_t b_n, int64_t m, int64_t n,
           int64_t k, float* c, int64_t ldc, int accumulate, float* part, hipStream_t s);

}  // namespace lpf
}  // namespace ts
