"""A key with NaN components leaves rows that do not see it as they are, where
its 64-key tile starts past the last key that their 32-row block sees (head dims
whose kernels pass over such tiles).  Bar: the fp32 reference of the same rows
over the keys they see, 2e-2 (16-bit inputs and outputs of size about 1)."""

from __future__ import annotations

import pytest
import torch

from oracle import attention as ref
from thundersync_amd import attention as hip

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("head_dim", [32, 64, 96, 192, 80])
@pytest.mark.parametrize("hq,hkv", [(2, 2), (4, 2), (4, 1)])
@pytest.mark.parametrize("where", ["key", "value"])
def test_nan_key_past_a_rows_reach(cuda, head_dim, hq, hkv, where):
    print(f"NaN {where} past the rows' reach: head dim {head_dim}, heads {hq}/{hkv}", flush=True)
    g = torch.Generator().manual_seed(head_dim + hq)
    # row r sees keys 0 .. 16 + r: the first block none past 47, the second some of the tile at 64
    rows, keys, seen = 128, 144, 32
    q, do = (torch.randn(rows, hq, head_dim, generator=g).bfloat16() for _ in range(2))
    k, v = (torch.randn(keys, hkv, head_dim, generator=g).bfloat16() for _ in range(2))
    (k if where == "key" else v)[64:] = float("nan")
    out_want, dq_want, *_ = ref.attention_with_grads(q[:seen], [k[: 16 + seen]], [v[: 16 + seen]], do[:seen], 0.1)
    leaves = [t.to(cuda).requires_grad_() for t in (q, k, v)]
    lay = hip.chain_layout(rows, [keys], hq, hkv)
    out, _ = hip.attention(leaves[0], lay, [leaves[1]], [leaves[2]], 0.1)
    dq, = torch.autograd.grad(out, leaves[:1], do.to(cuda))
    for got, want in ((out, out_want), (dq, dq_want)):
        assert (got[:seen].detach().float().cpu() - want).abs().max().item() <= 2e-2 * max(1.0, want.abs().max().item())
