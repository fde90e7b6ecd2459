"""RMSNorm kernels by vectors per lane.

The forward is built for 12, 20 and 24 vectors a lane beside the powers of two,
the backward for 10 and 12.  Each is met full, with its last vector part empty and with one
vector more than the variant below it.
"""

from __future__ import annotations

import pytest
import torch

from thundersync_amd.rms_norm import rms_norm_backward, rms_norm_forward

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("dtype", [torch.bfloat16, torch.float32])
@pytest.mark.parametrize("rows,width", [
    (1025, 2308), (1025, 3072), (1025, 4100), (1025, 5120), (1025, 5124), (1025, 6144), (1025, 6148),
    (16387, 4096)])
def test_forward_bytes(cuda, rows, width, dtype):
    print(f"rmsnorm fwd rows={rows} width={width} {dtype}", flush=True)
    g = torch.Generator(device=cuda).manual_seed(rows + width)
    x = torch.randn(rows, width, generator=g, device=cuda).to(dtype)
    w = torch.linspace(0.4, 3.0, width, device=cuda).to(dtype)
    y, rstd = rms_norm_forward(x, w, 1e-6)
    xf = x.float()
    want_rstd = torch.rsqrt(xf.pow(2).mean(-1, keepdim=True) + 1e-6)
    assert torch.equal(rstd, want_rstd) and torch.equal(y, w * (xf * want_rstd).to(dtype))


@pytest.mark.parametrize("dtype", [torch.bfloat16, torch.float32])
@pytest.mark.parametrize("rows,width", [(1, 4104), (9, 4104), (300, 5112), (2049, 5120), (300, 5128), (300, 6136),
                                        (7, 6144), (2049, 6144), (300, 6152), (33, 256), (40, 32)])
def test_backward(cuda, rows, width, dtype):
    print(f"rmsnorm bwd rows={rows} width={width} {dtype}", flush=True)
    g = torch.Generator(device=cuda).manual_seed(rows + width)
    x, dy = (torch.randn(rows, width, generator=g, device=cuda).to(dtype) for _ in range(2))
    w = torch.linspace(0.4, 3.0, width, device=cuda).to(dtype)
    rstd = torch.rsqrt(x.float().pow(2).mean(-1, keepdim=True) + 1e-6)
    dx, dw = rms_norm_backward(dy, x, w, rstd)
    xd, gd, r = x.double(), dy.double(), rstd.double()
    wg = w.double() * gd
    want_dx = r * wg - xd * r ** 3 * (wg * xd).mean(-1, keepdim=True)
    want_dw = (gd * xd * r).sum(0)
    # fp32 sums of `width` and `rows` terms, then one rounding to the dtype: half a unit
    # of it, and 2^-24 for each of the at most `n` additions into the sum of magnitudes
    unit = {torch.bfloat16: 2.0 ** -8, torch.float32: 2.0 ** -24}[dtype]
    slack_dx = 2.0 ** -24 * ((wg * xd).abs().mean(-1, keepdim=True) * 64 * xd.abs() * r ** 3 + 8 * (r * wg).abs()
                             + 8 * want_dx.abs())
    slack_dw = 2.0 ** -24 * (rows + 8) * (gd * xd * r).abs().sum(0)
    assert bool(((dx.double() - want_dx).abs() <= unit * want_dx.abs() + slack_dx).all())
    assert bool(((dw.double() - want_dw).abs() <= unit * want_dw.abs() + slack_dw).all())


@pytest.mark.parametrize("rows", [1024, 1025, 2048, 2049])
@pytest.mark.parametrize("width", [6148, 7168])
def test_forward_bytes_of_wide_fp32_rows(cuda, rows, width):
    """fp32 rows of 32 vectors: launches of 257 to 512 blocks of four rows load the weight
    after the reduction, the others beside the row."""
    test_forward_bytes(cuda, rows, width, torch.float32)


@pytest.mark.parametrize("dtype", [torch.bfloat16, torch.float16, torch.float32])
@pytest.mark.parametrize("rows,width", [(6147, 2308), (8192, 3072), (6147, 3076), (4099, 4096), (8192, 4096), (8195, 4096),
                                        (6145, 2048)])
def test_forward_bytes_around_one_round(cuda, rows, width, dtype):
    """Rows of 8 to 16 vectors a lane in launches that load the weight after the reduction
    (one round of the CUs then), and just past them."""
    test_forward_bytes(cuda, rows, width, dtype)


@pytest.mark.parametrize("rows,width", [(255 * 8, 512), (256 * 32, 512), (256 * 32 + 1, 1024), (2049, 1536)])
def test_backward_of_narrow_rows(cuda, rows, width):
    """Rows per block: one pass of its waves up to 256 blocks, 32 rows from there."""
    test_backward(cuda, rows, width, torch.bfloat16)
