"""The last token tile of the logprob GEMMs at every width it can take (64,
128, 192 or 256 tokens) and at its edges: values, the hidden gradient and the
weight gradient against a dense log-softmax in fp32 from the same 16-bit
inputs, with targets on the first and last vocabulary rows of tiles and out of
range.  Bars: logprob and entropy 1e-3 (the operator's), gradients 1e-2 of
their largest value (dlogits and results round to the element type, 2^-8 each,
and errors of a sum average out)."""

from __future__ import annotations

import pytest
import torch

from thundersync_amd import fused_logprob as fl

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("rows", [1, 63, 64, 65, 128, 129, 192, 193, 255, 256, 257, 320, 385, 449])
@pytest.mark.parametrize("dim,vocab,dtype", [(64, 700, torch.bfloat16), (200, 513, torch.float16)])
def test_widths_of_the_last_token_tile(cuda, rows, dim, vocab, dtype):
    print(f"narrow tiles rows={rows} dim={dim} vocab={vocab} {dtype}", flush=True)
    g = torch.Generator().manual_seed(rows + vocab)
    h0 = torch.randn(rows, dim, generator=g).to(dtype)
    w0 = (torch.randn(vocab, dim, generator=g) * 0.1).to(dtype)
    t = torch.randint(0, vocab, (rows,), generator=g)
    edges = torch.tensor([0, 31, 32, 63, 64, 127, 128, 255, 256, 511, vocab - 1])
    t[: len(edges)] = edges[:rows]
    bad = rows > 20
    if bad:
        t[15], t[16] = -1, vocab
    c_lp, c_ent = torch.randn(rows, generator=g), torch.randn(rows, generator=g)
    h, w = h0.to(cuda).requires_grad_(), w0.to(cuda).requires_grad_()
    lp, ent = fl.fused_logprob_entropy(h, w, t.to(cuda), chunk=256)
    torch.autograd.backward([lp, ent], [c_lp.to(cuda), c_ent.to(cuda)])
    hx, wx = h0.float().requires_grad_(), w0.float().requires_grad_()
    logp = torch.log_softmax(hx @ wx.t(), -1)
    valid = (t >= 0) & (t < vocab)
    lpx = logp.gather(1, t.clamp(0, vocab - 1)[:, None])[:, 0]
    entx = -(logp.exp() * logp).sum(-1)
    # an out-of-range target has no one-hot term: every vocabulary entry takes -p g_lp
    # there, the gradient of -logsumexp alone
    lse = torch.logsumexp(hx @ wx.t(), -1)
    ((torch.where(valid, lpx, -lse)) * c_lp + entx * c_ent).sum().backward()
    assert (lp.detach().cpu() - lpx.detach())[valid].abs().max().item() <= 1e-3
    assert bool(lp.detach().cpu()[~valid].isnan().all())
    assert (ent.detach().cpu() - entx.detach()).abs().max().item() <= 1e-3
    for got, want in ((h.grad, hx.grad), (w.grad, wx.grad)):
        assert (got.float().cpu() - want).abs().max().item() <= 1e-2 * want.abs().max().item()
