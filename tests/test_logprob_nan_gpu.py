"""A head row of NaN makes every logprob and entropy NaN, as a dense log-softmax
does, wherever in the vocabulary's last tile the row lies: the row may be the
only one that a lane of the kernels holds there.  (Plain comparison: the values
are NaN or not, no tolerance.)"""

from __future__ import annotations

import pytest
import torch

from thundersync_amd import fused_logprob as fl

pytestmark = pytest.mark.gpu

DTYPES = [torch.bfloat16, torch.float16, torch.float32]


@pytest.mark.parametrize("dtype", DTYPES)
@pytest.mark.parametrize("rows", [5, 100, 160, 300])
@pytest.mark.parametrize("past", [1, 5, 33, 65, 129, 193, 256])
def test_last_head_row_nan(cuda, dtype, rows, past):
    """`past`: vocabulary rows in the last tile of 256."""
    print(f"NaN head row: {dtype} rows={rows} past={past}", flush=True)
    g = torch.Generator().manual_seed(past)
    h, w = torch.randn(rows, 64, generator=g).to(dtype), torch.randn(256 + past, 64, generator=g).to(dtype)
    w[-1] = float("nan")
    t = torch.randint(0, 256, (rows,), generator=g)
    lp, ent = fl.fused_logprob_entropy(h.to(cuda), w.to(cuda), t.to(cuda))
    assert bool(lp.isnan().all()) and bool(ent.isnan().all())


@pytest.mark.parametrize("dtype", DTYPES)
def test_head_rows_that_score_minus_infinity(cuda, dtype):
    """Whole tiles of logits of -inf add nothing to the logprob."""
    print(f"-inf head rows: {dtype}", flush=True)
    g = torch.Generator().manual_seed(1)
    h, w = torch.randn(70, 64, generator=g), torch.randn(600, 64, generator=g) * 0.1
    h[:, 0], w[:, 0] = 1.0, 0.0
    w[128:512, 0] = float("-inf")
    h, w = h.to(dtype), w.to(dtype)
    t = torch.randint(0, 128, (70,), generator=g)
    lp = fl.fused_logprob(h.to(cuda), w.to(cuda), t.to(cuda))
    want = torch.log_softmax(h.double() @ w.double().t(), -1).gather(1, t[:, None])[:, 0]
    # 64 exact products summed in fp32 and log-sum-exp over 216 terms: the bars of the fp32 operator tests
    torch.testing.assert_close(lp.cpu().double(), want, rtol=1e-5, atol=1e-5)
