"""The weight gradient's last vocabulary row where the vocabulary is not a
multiple of 8: the last chunk of a dlogits row is whole in every token row,
those that end a stage of 32 tokens included."""

from __future__ import annotations

import pytest
import torch

from thundersync_amd import fused_logprob as fl

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("rows,vocab", [(33, 513), (32, 511), (64, 700), (1, 9), (289, 50257)])
def test_last_vocabulary_row(cuda, rows, vocab):
    print(f"odd vocabulary rows={rows} vocab={vocab}", flush=True)
    g = torch.Generator(device=cuda).manual_seed(rows)
    dim = 64
    h = torch.randn(rows, dim, generator=g, device=cuda).bfloat16().requires_grad_()
    w = (torch.randn(vocab, dim, generator=g, device=cuda) * 0.1).bfloat16().requires_grad_()
    t = torch.full((rows,), vocab - 1, device=cuda)
    fl.fused_logprob(h, w, t).sum().backward()
    hx, wx = h.detach().double(), w.detach().double()
    dl = torch.nn.functional.one_hot(t, vocab).double() - torch.softmax(hx @ wx.t(), -1)
    want = dl[:, -1] @ hx
    # dlogits and the result rounded to bf16 (half of 2^-7 each, of the sum of magnitudes), their
    # product and the fp32 logits' error in dlogits (1e-5 of it)
    bar = (2.0 ** -7 + 2.0 ** -16 + 1e-5) * (dl[:, -1].abs()[:, None] * hx.abs()).sum(0)
    assert bool(((w.grad[-1].double() - want).abs() <= bar).all())
