"""The fp32 matrix-instruction kernels of the fused logprob at the edges of
their tiles, against the host in fp64.

Tiles are 64 or 128 rows by 128 columns, K runs 32 at a time, and a product
whose tiles leave the device idle is cut into contraction ranges.  Bounds: a
sum of K fp32 products in any order is off by at most about K eps / 2 times
the sum of the magnitudes (eps = 2^-23), and by sqrt(K) eps of their root sum
of squares when the roundings are independent; the products are held to
4 sqrt(K) eps of the latter, the values to rtol 1e-5 / atol 1e-5 (the bars of
the fp32 operator tests, dims of this size).
"""

from __future__ import annotations

import math

import pytest
import torch

from thundersync_amd import _lib
from thundersync_amd import fused_logprob as fl

pytestmark = pytest.mark.gpu

EPS = 2.0 ** -23


@pytest.mark.parametrize("m,n,k,accumulate", [
    (1, 1, 1, False), (64, 128, 32, True), (65, 129, 33, False), (128, 127, 512, True),
    (63, 130, 2049, False), (200, 257, 1100, True), (1024, 160, 4099, False),
])
@pytest.mark.parametrize("a_kfast", [True, False])
@pytest.mark.parametrize("b_kfast", [True, False])
@pytest.mark.parametrize("pad", [0, 1])
def test_matmul_layouts(cuda, m, n, k, accumulate, a_kfast, b_kfast, pad):
    """Each operand K-contiguous or not, rows that are whole 16-byte vectors
    (pad 0, rounded up to 4) or not, with and without contraction ranges."""
    print(f"f32 product {m}x{n}x{k} a_kfast={a_kfast} b_kfast={b_kfast} pad={pad} acc={accumulate}", flush=True)
    g = torch.Generator().manual_seed(m + n + k)
    lib = _lib.require_library()

    def operand(rows, cols):  # [rows, cols] with a row stride that is (pad 0) or is not a multiple of 4
        ld = (cols + 3) // 4 * 4 + pad
        t = torch.randn(rows, ld, generator=g)
        return t[:, :cols], t.to(cuda)

    a, ad = operand(m, k) if a_kfast else operand(k, m)
    b, bd = operand(n, k) if b_kfast else operand(k, n)
    a_m, a_k = (ad.stride(0), 1) if a_kfast else (1, ad.stride(0))
    b_n, b_k = (bd.stride(0), 1) if b_kfast else (1, bd.stride(0))
    am = (a if a_kfast else a.t()).double()
    bm = (b.t() if b_kfast else b).double()
    c0 = torch.randn(m, n, generator=g) if accumulate else torch.zeros(m, n)
    want = am @ bm + c0.double()
    bound = 4 * math.sqrt(k + 1) * EPS * (am.square() @ bm.square() + c0.double().square()).sqrt()
    bytes_ = int(lib.ts_matmul_exact_workspace(m, n, k, 0))
    for ranges in ([False, True] if bytes_ else [False]):
        c = c0.to(cuda)
        ws = torch.empty(max(bytes_, 16), dtype=torch.uint8, device=cuda)
        _lib.check(lib.ts_matmul_exact_ws(ad.data_ptr(), a_m, a_k, bd.data_ptr(), b_k, b_n, m, n, k, c.data_ptr(), n,
                                          int(accumulate), ws.data_ptr() if ranges else None, bytes_, 0,
                                          _lib.stream_of(c)), "product")
        off = (c.cpu().double() - want).abs()
        assert bool((off <= bound + 1e-30).all()), float((off / bound).max())


@pytest.mark.parametrize("rows,dim,vocab", [
    (1, 4, 1), (1, 33, 129), (64, 32, 128), (65, 31, 127), (128, 64, 4096), (129, 100, 4097), (700, 36, 16500),
])
def test_values_and_gradients_at_tile_edges(cuda, rows, dim, vocab):
    print(f"f32 head rows={rows} dim={dim} vocab={vocab}", flush=True)
    g = torch.Generator().manual_seed(rows + vocab)
    h0, w0 = torch.randn(rows, dim, generator=g), torch.randn(vocab, dim, generator=g) * 0.1
    t = torch.randint(0, vocab, (rows,), generator=g)
    c_lp, c_ent = torch.randn(rows, generator=g), torch.randn(rows, generator=g)
    h, w = h0.to(cuda).requires_grad_(), w0.to(cuda).requires_grad_()
    lp, ent = fl.fused_logprob_entropy(h, w, t.to(cuda), chunk=256)
    (lp * c_lp.to(cuda) + ent * c_ent.to(cuda)).sum().backward()
    hx, wx = h0.double().requires_grad_(), w0.double().requires_grad_()
    logp = torch.log_softmax(hx @ wx.t(), -1)
    lpx = logp.gather(1, t[:, None])[:, 0]
    entx = -(logp.exp() * logp).sum(-1)
    (lpx * c_lp.double() + entx * c_ent.double()).sum().backward()
    torch.testing.assert_close(lp.detach().cpu().double(), lpx.detach(), rtol=1e-5, atol=1e-5)
    torch.testing.assert_close(ent.detach().cpu().double(), entx.detach(), rtol=1e-5, atol=1e-5)
    torch.testing.assert_close(h.grad.cpu().double(), hx.grad, rtol=1e-4, atol=1e-5)
    torch.testing.assert_close(w.grad.cpu().double(), wx.grad, rtol=1e-4, atol=1e-5)


def test_infinite_and_nan_logits(cuda):
    """Rows with a logit of -inf, +inf or NaN give what a dense log-softmax
    gives: a finite logprob and a NaN entropy, NaN, NaN; other rows are untouched."""
    print("f32 head with infinite and NaN logits", flush=True)
    g = torch.Generator().manual_seed(2)
    h, w = torch.randn(70, 8, generator=g), torch.randn(300, 8, generator=g)
    w[:, 0] = 0.0
    w[7, 0] = -1.0
    h[:, 0] = 0.0
    h[3, 0], h[5, 0], h[9, 1] = math.inf, -math.inf, math.nan
    # 0 * inf is NaN: keep the infinite feature on the one row that reads it
    dense = (h.double() @ w.double().t())
    t = torch.full((70,), 11)
    lp, ent = fl.fused_logprob_entropy(h.to(cuda), w.to(cuda), t.to(cuda))
    logp = torch.log_softmax(dense, -1)
    want = logp[:, 11]
    went = -(logp.exp() * logp).sum(-1)
    torch.testing.assert_close(lp.cpu().double(), want, rtol=1e-5, atol=1e-5, equal_nan=True)
    torch.testing.assert_close(ent.cpu().double(), went, rtol=1e-5, atol=1e-5, equal_nan=True)
