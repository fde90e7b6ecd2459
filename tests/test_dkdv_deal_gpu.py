"""dK/dV at head dim 128 over both item sizes, whatever the GQA group: the
kernel that deals (head, row block) steps to its waves (48-key items) and the
key-split kernel (64-key items), against the fp32 oracle and, on the dS route,
through dQ; segments shorter than the four waves' blocks, runs with several
visits, visits that see only part of a run, remainders of the key block."""

from __future__ import annotations

import pytest
import torch

from oracle import attention as ref
from thundersync_amd import attention as hip

pytestmark = pytest.mark.gpu

CASES = [
    # hq, hkv, prompt keys, [(own rows)] -- every segment reads the prompt and its own rows
    (5, 1, 1, [1]),
    (6, 2, 47, [31, 33]),
    (3, 1, 49, [65, 1, 32]),
    (10, 2, 130, [5, 200, 64, 7, 129]),
    (4, 4, 96, [33, 160]),
    (8, 2, 64, [40, 100]),
]


@pytest.mark.parametrize("kv_block", [48, 64])
@pytest.mark.parametrize("ds", ["auto", "off"])
@pytest.mark.parametrize("case", range(len(CASES)))
def test_dealt_and_key_split_items(cuda, monkeypatch, case, ds, kv_block):
    hq, hkv, prompt, rows = CASES[case]
    print(f"dkdv items of {kv_block} keys, {hq}/{hkv} heads, prompt {prompt}, rows {rows}, ds {ds}", flush=True)
    monkeypatch.setenv(hip.DS_ENV, ds)
    monkeypatch.setattr(hip.AttnLayout, "call_kv_block", lambda self, device, head_dim: kv_block)
    g = torch.Generator().manual_seed(case)
    d, total = 128, sum(rows)
    q, do = (torch.randn(total, hq, d, generator=g).to(torch.bfloat16) for _ in range(2))
    ks = [torch.randn(n, hkv, d, generator=g).to(torch.bfloat16) for n in (prompt, *rows)]
    vs = [torch.randn(n, hkv, d, generator=g).to(torch.bfloat16) for n in (prompt, *rows)]
    runs = tuple(hip.Run(i, 0, n) for i, n in enumerate((prompt, *rows)))
    seg_q, at = [], 0
    for n in rows:
        seg_q.append((at, n))
        at += n
    lay = hip.AttnLayout(q_rows=total, hq=hq, hkv=hkv, source_rows=(prompt, *rows), runs=runs, seg_q=tuple(seg_q),
                         seg_spans=tuple(((0, 0), (i + 1, prompt)) for i in range(len(rows))))
    qc = q.to(cuda).requires_grad_()
    kc = [k.to(cuda).requires_grad_() for k in ks]
    vc = [v.to(cuda).requires_grad_() for v in vs]
    hip.attention(qc, lay, kc, vc, d ** -0.5)[0].backward(do.to(cuda))
    want_k, want_v = [torch.zeros(k.shape) for k in ks], [torch.zeros(v.shape) for v in vs]
    want_q = torch.zeros(q.shape)
    for i, (a, n) in enumerate(seg_q):
        _, dq, dk, dv = ref.attention_with_grads(q[a:a + n], [ks[0], ks[i + 1]], [vs[0], vs[i + 1]], do[a:a + n],
                                                 d ** -0.5)
        want_q[a:a + n] = dq
        for j, s in enumerate((0, i + 1)):
            want_k[s] += dk[j]
            want_v[s] += dv[j]
    for got, want in zip((qc.grad, *(k.grad for k in kc), *(v.grad for v in vc)), (want_q, *want_k, *want_v)):
        # the bar of the attention gradients: 2e-2 of the largest value (at least 1)
        assert (got.float().cpu() - want).abs().max().item() <= 2e-2 * max(1.0, want.abs().max().item())
