"""Work items cut into parts (forward and the dS route's dQ pass) at head dims
128 and 256: any part count -- more parts than tiles, parts that see nothing of
some rows, part edges inside and between runs -- against whole items and the
fp32 oracle.  A part's probabilities are taken against its own reference point
before they are rounded to bf16, so each of them may round differently: by at
most 2^-8 of itself, which moves an output, a weighted mean of values, by at
most 2^-8 max |v|, and its own rounding by 2^-8 of it.  lse comes from the
unrounded sums (1e-5); gradients keep the oracle's bar, 2e-2 of their largest
value (at least 1)."""

from __future__ import annotations

import pytest
import torch

from oracle import attention as ref
from thundersync_amd import _lib
from thundersync_amd import attention as hip

pytestmark = pytest.mark.gpu


class _Parts:
    """The library with fixed part counts."""

    def __init__(self, lib, parts):
        self._lib, self._parts = lib, parts

    def __getattr__(self, name):
        if name in ("ts_attn_fwd_parts", "ts_attn_dq_parts"):
            return lambda *args: self._parts
        return getattr(self._lib, name)


def run(cuda, layout, q, ks, vs, do, parts, monkeypatch):
    lib = _lib.require_library()
    with monkeypatch.context() as m:
        m.setattr(_lib, "_LIB", _Parts(lib, parts))
        qc = q.to(cuda).requires_grad_()
        kc, vc = ([t.to(cuda).requires_grad_() for t in x] for x in (ks, vs))
        out, lse = hip.attention(qc, layout, kc, vc, q.shape[2] ** -0.5)
        out.backward(do.to(cuda))
        torch.cuda.synchronize()
    return out.detach(), lse, qc.grad, [k.grad for k in kc]


@pytest.mark.parametrize("d,hq,hkv", [(128, 8, 2), (128, 5, 1), (128, 4, 2), (256, 6, 1), (256, 4, 1)])
@pytest.mark.parametrize("rows,chunks", [([1], [[1]]), ([1], [[70, 1]]), ([33], [[512, 31, 33]]),
                                         ([65, 5, 130], [[64, 65], [1, 5], [300, 17, 130]])])
def test_parts_equal_whole_items(cuda, monkeypatch, d, hq, hkv, rows, chunks):
    print(f"parts d={d} heads {hq}/{hkv} rows={rows} chunks={chunks}", flush=True)
    g = torch.Generator().manual_seed(d + hq + sum(rows))
    total = sum(rows)
    q, do = (torch.randn(total, hq, d, generator=g).to(torch.bfloat16) for _ in range(2))
    lens = [n for c in chunks for n in c]
    ks, vs = ([torch.randn(n, hkv, d, generator=g).to(torch.bfloat16) for n in lens] for _ in range(2))
    spans, run0, seg_q, at = [], 0, [], 0
    for n, c in zip(rows, chunks):
        pos, sp = 0, []
        for j, m in enumerate(c):
            sp.append((run0 + j, pos))
            pos += m
        run0 += len(c)
        spans.append(tuple(sp))
        seg_q.append((at, n))
        at += n
    layout = hip.AttnLayout(q_rows=total, hq=hq, hkv=hkv, source_rows=tuple(lens),
                            runs=tuple(hip.Run(i, 0, n) for i, n in enumerate(lens)), seg_q=tuple(seg_q),
                            seg_spans=tuple(spans))
    whole = run(cuda, layout, q, ks, vs, do, 1, monkeypatch)
    run0 = 0
    for (a, n), c in zip(seg_q, chunks):
        o, dq, _, _ = ref.attention_with_grads(q[a:a + n], ks[run0:run0 + len(c)], vs[run0:run0 + len(c)],
                                               do[a:a + n], d ** -0.5)
        run0 += len(c)
        for got, want in ((whole[0][a:a + n], o), (whole[2][a:a + n], dq)):
            assert (got.float().cpu() - want).abs().max().item() <= 2e-2 * max(1.0, want.abs().max().item())
    for parts in (2, 3, 7, 32):
        got = run(cuda, layout, q, ks, vs, do, parts, monkeypatch)
        off = (got[0].float() - whole[0].float()).abs()
        most = max(v.float().abs().max().item() for v in vs)
        assert bool((off <= 2 ** -8 * (most + whole[0].float().abs())).all()), (parts, off.max().item())
        torch.testing.assert_close(got[1], whole[1], rtol=1e-5, atol=1e-5)
        for x, y in zip([got[2], *got[3]], [whole[2], *whole[3]]):
            assert (x.float() - y.float()).abs().max().item() <= 2e-2 * max(1.0, y.float().abs().max().item())
        again = run(cuda, layout, q, ks, vs, do, parts, monkeypatch)
        assert all(torch.equal(a, b) for a, b in zip(got[:3], again[:3]))


def test_refused_parts(cuda):
    """A workspace that is missing or too small, and head dims whose kernels do not split, are errors."""
    lib = _lib.require_library()
    import ctypes

    for d, parts, floats in ((128, 2, 0), (128, 2, 2 * 4 * 8 * 130 - 1), (64, 2, 1 << 20), (128, 0, 0)):
        lay = hip.chain_layout(8, [8], 4, 1)
        q = torch.zeros(8, 4, d, dtype=torch.bfloat16, device=cuda)
        k = torch.zeros(8, 1, d, dtype=torch.bfloat16, device=cuda)
        lse = torch.zeros(4, 8, device=cuda)
        _, (runs, _, keep) = lay._upload(q.device, 48, hip._gather(lay, q, [k], [k]))
        problem = lay.problem(q.device, runs, 0.1, q.dtype, d, 48)
        ws = torch.zeros(max(floats, 4), device=cuda)
        status = lib.ts_attn_fwd_split(ctypes.byref(problem), hip._rows(q), hip._rows(q.clone()), lse.data_ptr(), 8,
                                       parts, ws.data_ptr() if floats else None, floats * 4, _lib.stream_of(q))
        assert status != 0 and "parts" in lib.ts_hip_last_error().decode()
    torch.cuda.synchronize()
