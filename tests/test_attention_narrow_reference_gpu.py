"""The softmax reference point at head dims 32, 64, 96 and 192: a row's running
maximum, exactly.  The largest weight of a row is then 1 and loses nothing when
the weights are rounded to the element type; scores of any size, and scales of
zero and below it, keep their softmax."""

from __future__ import annotations

import pytest
import torch

from oracle import attention as ref
from thundersync_amd import attention as hip

pytestmark = pytest.mark.gpu

DIMS = [32, 64, 96, 192]
HALF_UNIT = {torch.bfloat16: 2.0 ** -9, torch.float16: 2.0 ** -12}  # of a number in [1, 2), relative to 2


@pytest.mark.parametrize("dtype", [torch.bfloat16, torch.float16])
@pytest.mark.parametrize("dim", DIMS)
@pytest.mark.parametrize("late", [33, 70, 127])
def test_largest_weight_is_exact(cuda, dim, late, dtype):
    """Every key scores 0 but key `late`, whose score is in (0, 5.5) and whose
    value alone is not zero: the output is that key's weight over the fp32 sum of
    all weights, rounded once."""
    print(f"largest weight: head dim {dim} {dtype}, key {late}", flush=True)
    g = torch.Generator().manual_seed(dim + late)
    rows, keys, hq, scale = 200, 400, 4, 1.0
    q = torch.zeros(rows, hq, dim)
    q[..., 0] = 0.05 + 5.4 * torch.rand(rows, hq, generator=g)
    k, v = torch.zeros(keys, 2, dim), torch.zeros(keys, 2, dim)
    k[late, :, 0] = 1.0
    v[late] = 1.0
    q, k, v = (t.to(dtype) for t in (q, k, v))
    out, _ = hip.attention(q.to(cuda), hip.chain_layout(rows, [keys], hq, 2), [k.to(cuda)], [v.to(cuda)], scale)
    want, _ = ref.bottom_right_attention(q, k, v, scale, dtype=torch.float64)
    off = (out.double().cpu() - want).abs()
    # one rounding of the result (half a unit in the last place, at most 2^-9 or 2^-12 times twice
    # it) and the fp32 exponential, sum and division (under 2^-18)
    bar = (2 * HALF_UNIT[dtype] + 2.0 ** -18) * want
    assert bool((off <= bar).all()), float((off / bar).max())


@pytest.mark.parametrize("dim", DIMS)
@pytest.mark.parametrize("size", [1e4, 1e10, 1e25])
def test_scores_of_any_size(cuda, dim, size):
    """Scores of the order of `size`, far apart: each row takes the value of its
    best key."""
    print(f"scores of {size}: head dim {dim}", flush=True)
    g = torch.Generator().manual_seed(dim)
    rows, keys = 50, 150
    q, k = torch.zeros(rows, 2, dim), torch.zeros(keys, 1, dim)
    q[..., 0] = torch.where(torch.rand(rows, 2, generator=g) < 0.5, -1.0, 1.0)
    k[:, 0, 0] = size * (torch.randperm(keys, generator=g) - keys // 2)
    v = torch.randn(keys, 1, dim, generator=g)
    q, k, v = (t.bfloat16() for t in (q, k, v))
    # keys of equal bf16 scores share a row's weight: the softmax of the rounded keys
    out, _ = hip.attention(q.to(cuda), hip.chain_layout(rows, [keys], 2, 1), [k.to(cuda)], [v.to(cuda)], 1.0)
    want, _ = ref.bottom_right_attention(q, k, v, 1.0, dtype=torch.float64)
    off = (out.double().cpu() - want).abs()
    assert bool((off <= 2e-2 * max(1.0, want.abs().max().item())).all()), float(off.max())


@pytest.mark.parametrize("dim", DIMS)
@pytest.mark.parametrize("scale", [0.0, -0.125])
def test_scales_of_zero_and_below(cuda, dim, scale):
    print(f"scale {scale}: head dim {dim}", flush=True)
    g = torch.Generator().manual_seed(dim)
    rows, lens = 70, (33, 90)
    q, do = (torch.randn(rows, 4, dim, generator=g).bfloat16() for _ in range(2))
    ks, vs = ([torch.randn(n, 2, dim, generator=g).bfloat16() for n in lens] for _ in range(2))
    qc = q.to(cuda).requires_grad_()
    kc, vc = ([t.to(cuda).requires_grad_() for t in x] for x in (ks, vs))
    out, _ = hip.attention(qc, hip.chain_layout(rows, lens, 4, 2), kc, vc, scale)
    out.backward(do.to(cuda))
    want_o, want_q, want_k, want_v = ref.attention_with_grads(q, ks, vs, do, scale, dtype=torch.float64)
    for got, want in ((out, want_o), (qc.grad, want_q), *zip((k.grad for k in kc), want_k),
                      *zip((v.grad for v in vc), want_v)):
        off = (got.detach().double().cpu() - want).abs()
        assert bool((off <= 2e-2 * max(1.0, want.abs().max().item())).all()), float(off.max())
