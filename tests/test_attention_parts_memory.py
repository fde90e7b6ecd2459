"""The workspace of work items cut into parts: bounded by what the items cover,
not by the rows of the query they lie in, and done without where the device has
no memory for it."""

from __future__ import annotations

import ctypes

import pytest
import torch

from oracle import attention as ref
from thundersync_amd import _lib
from thundersync_amd import attention as hip


def sparse(rows, hq, hkv, at=0, own=48, context=4096):
    """One segment of `own` rows at row `at` of a query of `rows` rows."""
    return hip.AttnLayout(q_rows=rows, hq=hq, hkv=hkv, source_rows=(context, own),
                          runs=(hip.Run(0, 0, context), hip.Run(1, 0, own)), seg_q=((at, own),),
                          seg_spans=(((0, 0), (1, context)),))


@pytest.mark.skipif(_lib.library() is None, reason="libthundersync_hip.so not built")
@pytest.mark.parametrize("dim,hq,hkv", [(128, 32, 8), (128, 40, 8), (256, 24, 4)])
def test_workspace_follows_the_items(dim, hq, hkv):
    lib, cpu = _lib.require_library(), torch.device("cpu")
    sizes = []
    for rows in (48, 65536):
        lay = sparse(rows, hq, hkv)
        kvb = lay.call_kv_block(cpu, dim)
        problem = lay.problem(cpu, 0, 0.1, torch.bfloat16, dim, kvb)
        tabs = lay.device_tables(cpu, kvb)
        n_dq = tabs["n_dq_work"] if dim == 128 else 0
        keys = lay._description()["max_keys"]
        fwd, dq = lib.ts_attn_fwd_parts(ctypes.byref(problem), keys), lib.ts_attn_dq_parts(
            ctypes.byref(problem), n_dq, keys)
        assert fwd > 1 and dq > 1
        sizes.append((lib.ts_attn_fwd_parts_workspace(ctypes.byref(problem), fwd),
                      lib.ts_attn_dq_parts_workspace(ctypes.byref(problem), n_dq, dq)))
        # one part of one item and head chunk: 128 (row, head) slots, 256 for the 64-row items
        assert lib.ts_attn_fwd_parts_workspace(ctypes.byref(problem), 1) == 0
    (fwd, dq), (fwd_sparse, dq_sparse) = sizes
    # the same items: at most the slots of half-empty items more
    assert 0 < fwd_sparse <= 3 * fwd <= 256 << 20
    assert 0 < dq_sparse <= 3 * dq <= 256 << 20


@pytest.mark.gpu
@pytest.mark.parametrize("dim,hq,hkv", [(128, 8, 2), (128, 5, 1), (256, 6, 1)])
@pytest.mark.parametrize("workspace", [True, False])
def test_sparse_segment_in_parts(cuda, monkeypatch, dim, hq, hkv, workspace):
    print(f"sparse segment: head dim {dim}, {hq}/{hkv} heads, workspace {workspace}", flush=True)
    if not workspace:
        monkeypatch.setattr(hip, "_parts_workspace", lambda nbytes, device: None)
    g = torch.Generator().manual_seed(dim + hq)
    rows, at, own, context = 3000, 1234, 70, 2500
    lay = sparse(rows, hq, hkv, at, own, context)
    q, do = (torch.randn(rows, hq, dim, generator=g).bfloat16() for _ in range(2))
    ks, vs = ([torch.randn(n, hkv, dim, generator=g).bfloat16() for n in (context, own)] for _ in range(2))
    qc = q.to(cuda).requires_grad_()
    kc, vc = ([t.to(cuda).requires_grad_() for t in x] for x in (ks, vs))
    out, _ = hip.attention(qc, lay, kc, vc, dim ** -0.5)
    out.backward(do.to(cuda))
    want = ref.attention_with_grads(q[at:at + own], ks, vs, do[at:at + own], dim ** -0.5)
    for got, w in ((out[at:at + own], want[0]), (qc.grad[at:at + own], want[1]),
                   *zip((k.grad for k in kc), want[2]), *zip((v.grad for v in vc), want[3])):
        assert (got.float().cpu() - w).abs().max().item() <= 2e-2 * max(1.0, w.abs().max().item())
    assert bool((qc.grad[:at] == 0).all()) and bool((qc.grad[at + own:] == 0).all())


@pytest.mark.gpu
def test_memory_of_a_sparse_segment(cuda):
    """48 rows over 4144 keys in a query of 65536 rows: the call's own tensors and no gigabytes beside them."""
    print("memory of a sparse segment", flush=True)
    hq, hkv, dim, rows = 32, 8, 128, 65536
    lay = sparse(rows, hq, hkv)
    q = torch.zeros(rows, hq, dim, dtype=torch.bfloat16, device=cuda).requires_grad_()
    ks, vs = ([torch.zeros(n, hkv, dim, dtype=torch.bfloat16, device=cuda).requires_grad_() for n in (4096, 48)]
              for _ in range(2))
    torch.cuda.synchronize()
    torch.cuda.reset_peak_memory_stats()
    before = torch.cuda.memory_allocated()
    out, _ = hip.attention(q, lay, ks, vs, 0.1)
    out.backward(torch.zeros_like(out))
    torch.cuda.synchronize()
    # out, its gradient and dQ (512 MiB each), lse and the row statistics (24 MiB), and under 512 MiB
    assert torch.cuda.max_memory_allocated() - before < 3 * (512 << 20) + (24 << 20) + (512 << 20)
