"""Rows whose leading keys all score -inf beside rows of the same block that
have finite scores there: each row's output is its own softmax, over whole
items and items cut into parts.  Against a softmax in fp64 of the scores taken
to fp32's range (a product past it is -inf, as it is in the kernels)."""

from __future__ import annotations

import pytest
import torch

from oracle import attention as ref
from tests.test_attention_parts_gpu import _Parts
from thundersync_amd import _lib
from thundersync_amd import attention as hip

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("leading", [32, 45, 64, 100])
@pytest.mark.parametrize("dim,parts", [(32, 1), (64, 1), (96, 1), (192, 1), (128, 1), (256, 1), (128, 3), (256, 3)])
@pytest.mark.parametrize("hq,hkv", [(4, 1), (2, 1), (3, 3)])
def test_leading_keys_of_minus_infinity(cuda, monkeypatch, hq, hkv, dim, parts, leading):
    print(f"infinite scores: head dim {dim}, {hq}/{hkv} heads, {parts} parts, {leading} leading keys", flush=True)
    lib = _lib.require_library()
    monkeypatch.setattr(_lib, "_LIB", _Parts(lib, parts))
    g = torch.Generator().manual_seed(dim + leading)
    rows, keys, scale = 40, 200, dim ** -0.5
    q = torch.randn(rows, hq, dim, generator=g).bfloat16()
    k, v = (torch.randn(keys, hkv, dim, generator=g).bfloat16() for _ in range(2))
    # the leading keys' component 0 is the most negative bf16 value: rows with 4 there
    # reach -inf, rows with 2^-122 finite scores of -64, rows with 0 ordinary ones
    q[:, :, 0] = torch.tensor([4.0, 2.0 ** -122, 4.0, 0.0, 4.0]).repeat(rows // 5)[:, None].bfloat16()
    k[:, :, 0] = 0.0
    k[:leading, :, 0] = torch.finfo(torch.bfloat16).min
    out, lse = hip.attention(q.to(cuda), hip.chain_layout(rows, [keys], hq, hkv), [k.to(cuda)], [v.to(cuda)], scale)
    kx, vx = (t.double().repeat_interleave(hq // hkv, 1) for t in (k, v))
    scores = torch.einsum("qhd,khd->hqk", q.double(), kx)
    scores = torch.where(scores < -3.4028235e38, -torch.inf, scores) * scale
    scores = scores.masked_fill(torch.arange(keys) > keys - rows + torch.arange(rows)[:, None], -torch.inf)
    want = torch.einsum("hqk,khd->qhd", scores.softmax(-1), vx)
    off = (out.double().cpu() - want).abs()
    assert bool((off <= 2e-2 * max(1.0, want.abs().max().item())).all())
    torch.testing.assert_close(lse.double().cpu(), scores.logsumexp(-1), rtol=1e-5, atol=1e-4)


@pytest.mark.parametrize("dim", [32, 64, 96, 192])
@pytest.mark.parametrize("rows", [1, 40, 64])
def test_gradients_of_a_key_that_no_row_sees(cuda, dim, rows):
    """A key of -inf in a component that every query holds positive: its weight is
    0 in every row, and its own gradients are 0, in row blocks of 32 and in a
    remainder (whose missing rows are zeros: 0 * -inf is no score)."""
    print(f"a key of -inf: head dim {dim}, {rows} rows", flush=True)
    g = torch.Generator().manual_seed(dim + rows)
    q, do = (torch.randn(rows, 4, dim, generator=g) for _ in range(2))
    q[:, :, 0] = q[:, :, 0].abs() + 0.1
    k, v = (torch.randn(90, 2, dim, generator=g) for _ in range(2))
    k[17, :, 0] = -torch.inf
    q, do, k, v = (t.bfloat16() for t in (q, do, k, v))
    qc, kc, vc = (t.to(cuda).requires_grad_() for t in (q, k, v))
    out, _ = hip.attention(qc, hip.chain_layout(rows, [90], 4, 2), [kc], [vc], dim ** -0.5)
    out.backward(do.to(cuda))
    want_o, _, want_k, want_v = ref.attention_with_grads(q, [k], [v], do, dim ** -0.5, dtype=torch.float64)
    assert bool((want_k[0][17] == 0).all()) and bool((want_v[0][17] == 0).all())
    for got, want in ((out, want_o), (kc.grad, want_k[0]), (vc.grad, want_v[0])):
        off = (got.detach().double().cpu() - want).abs()
        assert bool((off <= 2e-2 * max(1.0, want.abs().max().item())).all())
