"""Gradients where runs end inside a key tile and every score is far below zero.

A key tile past the end of a run holds zero rows, whose score is 0: beside
scores around -26 (fp16) or -100 (bf16) its probability would be exp(26) or
exp(100), and dS past the range of the element type.  Q and K carry a constant
component, as a projection's bias gives them, that shifts every score; the runs
before the last one end at 70, 1, 31 and 65 keys.  Every kernel head dim, the
dQ kernels that recompute the scores (the dS route off at 128 and 256) and the
dS route, against the oracle in fp64."""

from __future__ import annotations

import pytest
import torch

from oracle import attention as ref
from thundersync_amd import attention as hip

pytestmark = pytest.mark.gpu

SHIFT = {torch.float16: 26.0, torch.bfloat16: 100.0}


@pytest.mark.parametrize("dtype", [torch.float16, torch.bfloat16])
@pytest.mark.parametrize("hq,hkv,runs,rows", [(2, 1, (70,), 40), (4, 1, (1, 31, 65), 130), (3, 3, (95, 33), 33)])
@pytest.mark.parametrize("dim,ds", [(32, "auto"), (64, "auto"), (96, "auto"), (192, "auto"), (128, "off"),
                                    (256, "off"), (128, "auto"), (256, "auto")])
def test_low_scores_beside_run_ends(cuda, monkeypatch, dim, ds, hq, hkv, runs, rows, dtype):
    print(f"run ends: head dim {dim} ds {ds} {dtype}, {hq}/{hkv} heads, runs {runs}, rows {rows}", flush=True)
    monkeypatch.setenv(hip.DS_ENV, ds)
    g = torch.Generator().manual_seed(dim + rows)
    scale, keys_const = dim ** -0.5, 4.0
    q, do = (torch.randn(rows, hq, dim, generator=g) for _ in range(2))
    q[..., 0] = -SHIFT[dtype] / (scale * keys_const)
    q, do = q.to(dtype), do.to(dtype)
    lens = (*runs, rows)
    ks, vs = ([torch.randn(n, hkv, dim, generator=g) for n in lens] for _ in range(2))
    for k in ks:
        k[..., 0] = keys_const
    ks, vs = [k.to(dtype) for k in ks], [v.to(dtype) for v in vs]
    qc = q.to(cuda).requires_grad_()
    kc, vc = ([t.to(cuda).requires_grad_() for t in x] for x in (ks, vs))
    out, _ = hip.attention(qc, hip.chain_layout(rows, lens, hq, hkv), kc, vc, scale)
    out.backward(do.to(cuda))
    want_o, want_q, want_k, want_v = ref.attention_with_grads(q, ks, vs, do, scale, dtype=torch.float64)
    # the bar of the attention outputs and gradients, 2e-2 of the largest value (at least 1); in the
    # constant column dS is multiplied by the constant, and the rounding errors of dS with it
    for got, want, const in ((out, want_o, 1.0), (qc.grad, want_q, keys_const),
                             *((k.grad, w, q[0, 0, 0].abs().item()) for k, w in zip(kc, want_k)),
                             *((v.grad, w, 1.0) for v, w in zip(vc, want_v))):
        off = (got.detach().double().cpu() - want).abs()
        off[..., 0] /= const
        bar = 2e-2 * max(1.0, want[..., 1:].abs().max().item())
        assert bool((off <= bar).all()), (off.max().item(), bar)
