"""The tile staging of head dims 32, 64, 96 and 192 at the edges of its tiles
(32 query rows, 48 or 64 keys), for every work split of the GQA groups, rows of
a stride above the heads, and with NaN in the memory right after every
sequence's rows and beside every row's heads: a tile reads its rows and nothing
past them.  Against the fp32 oracle."""

from __future__ import annotations

import pytest
import torch

from oracle import attention as ref
from thundersync_amd import attention as hip

pytestmark = pytest.mark.gpu

CASES = [
    # hq, hkv, prompt keys, own rows of each segment
    (4, 4, 1, [1]),
    (3, 1, 63, [31, 65]),
    (4, 2, 64, [33, 1, 128]),
    (6, 1, 65, [64, 97]),
    (8, 2, 47, [32, 130, 5]),
    (8, 1, 200, [260]),
]


def inside(values: torch.Tensor, device) -> torch.Tensor:
    """`values` [n, h, d] as a view of a larger NaN-filled tensor."""
    n, h, d = values.shape
    outer = torch.full((n + 70, h + 1, d), float("nan"), dtype=values.dtype, device=device)
    outer[:n, :h] = values.to(device)
    return outer[:n, :h]


@pytest.mark.parametrize("dtype", [torch.bfloat16, torch.float16])
@pytest.mark.parametrize("kv_block", [48, 64])
@pytest.mark.parametrize("dim", [32, 64, 96, 192])
@pytest.mark.parametrize("case", range(len(CASES)))
def test_tiles(cuda, monkeypatch, case, dim, kv_block, dtype):
    hq, hkv, prompt, rows = CASES[case]
    print(f"head dim {dim} {dtype}, items of {kv_block} keys, {hq}/{hkv} heads, prompt {prompt}, rows {rows}", flush=True)
    monkeypatch.setattr(hip.AttnLayout, "call_kv_block", lambda self, device, head_dim: kv_block)
    g = torch.Generator().manual_seed(10 * case + dim)
    total = sum(rows)
    q, do = (torch.randn(total, hq, dim, generator=g).to(dtype) for _ in range(2))
    ks = [torch.randn(n, hkv, dim, generator=g).to(dtype) for n in (prompt, *rows)]
    vs = [torch.randn(n, hkv, dim, generator=g).to(dtype) for n in (prompt, *rows)]
    seg_q, at = [], 0
    for n in rows:
        seg_q.append((at, n))
        at += n
    lay = hip.AttnLayout(q_rows=total, hq=hq, hkv=hkv, source_rows=(prompt, *rows),
                         runs=tuple(hip.Run(i, 0, n) for i, n in enumerate((prompt, *rows))), seg_q=tuple(seg_q),
                         seg_spans=tuple(((0, 0), (i + 1, prompt)) for i in range(len(rows))))
    qc = inside(q, cuda).detach().requires_grad_()
    kc = [inside(k, cuda).detach().requires_grad_() for k in ks]
    vc = [inside(v, cuda).detach().requires_grad_() for v in vs]
    out = hip.attention(qc, lay, kc, vc, dim ** -0.5)[0]
    out.backward(inside(do, cuda))
    want_o, want_q = torch.zeros(q.shape), torch.zeros(q.shape)
    want_k, want_v = [torch.zeros(k.shape) for k in ks], [torch.zeros(v.shape) for v in vs]
    for i, (a, n) in enumerate(seg_q):
        o, dq, dk, dv = ref.attention_with_grads(q[a:a + n], [ks[0], ks[i + 1]], [vs[0], vs[i + 1]], do[a:a + n],
                                                 dim ** -0.5)
        want_o[a:a + n], want_q[a:a + n] = o, dq
        for j, s in enumerate((0, i + 1)):
            want_k[s] += dk[j]
            want_v[s] += dv[j]
    for got, want in zip((out, qc.grad, *(k.grad for k in kc), *(v.grad for v in vc)),
                         (want_o, want_q, *want_k, *want_v)):
        # the bar of the attention outputs and gradients: 2e-2 of the largest value (at least 1)
        err = (got.detach().float().cpu() - want).abs()
        assert bool((err <= 2e-2 * max(1.0, want.abs().max().item())).all())
