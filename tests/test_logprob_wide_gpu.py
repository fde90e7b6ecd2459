"""The 320-token tiles of the logprob GEMMs (one tile where 256-token ones need
two, two where they need three) against a dense log-softmax in fp32 from the
same 16-bit inputs: rows at the tiles' edges, a ragged last vocabulary tile,
targets at the edges of vocabulary tiles and of the tokens' halves.  Bars as for
the narrow tiles: logprob and entropy 1e-3, gradients 1e-2 of their largest
value (dlogits and results round to the element type, 2^-8 each, and errors of a
sum average out)."""

from __future__ import annotations

import pytest
import torch

from thundersync_amd import fused_logprob as fl

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("rows,vocab,dtype", [
    (257, 66001, torch.bfloat16), (281, 66001, torch.float16), (320, 66001, torch.bfloat16),
    (321, 66001, torch.bfloat16), (600, 50257, torch.bfloat16), (640, 50257, torch.float16)])
def test_wide_tiles(cuda, rows, vocab, dtype):
    dim = 4096
    print(f"wide tiles rows={rows} vocab={vocab} {dtype}", flush=True)
    g = torch.Generator(device=cuda).manual_seed(rows)
    h = torch.randn(rows, dim, generator=g, device=cuda).to(dtype).requires_grad_()
    w = (torch.randn(vocab, dim, generator=g, device=cuda) * 0.02).to(dtype).requires_grad_()
    t = torch.randint(0, vocab, (rows,), generator=g, device=cuda)
    edges = torch.tensor([0, 31, 32, 63, 64, 255, 256, vocab - 1], device=cuda)
    for at in (0, 156, rows - 8):
        t[at:at + 8] = edges
    c_lp, c_ent = (torch.randn(rows, generator=g, device=cuda) for _ in range(2))
    lp, ent = fl.fused_logprob_entropy(h, w, t)
    torch.autograd.backward([lp, ent], [c_lp, c_ent])
    hx, wx = h.detach().float().requires_grad_(), w.detach().float().requires_grad_()
    logp = torch.log_softmax(hx @ wx.t(), -1)
    lpx = logp.gather(1, t[:, None])[:, 0]
    entx = -(logp.exp() * logp).sum(-1)
    (lpx * c_lp + entx * c_ent).sum().backward()
    assert (lp - lpx).abs().max().item() <= 1e-3
    assert (ent - entx).abs().max().item() <= 1e-3
    for got, want in ((h.grad, hx.grad), (w.grad, wx.grad)):
        assert (got.float() - want).abs().max().item() <= 1e-2 * want.abs().max().item()
