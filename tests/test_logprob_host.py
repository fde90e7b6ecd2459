"""Host side of the fused logprob (CPU): which operands the kernels read in place."""

from __future__ import annotations

import torch

from thundersync_amd import fused_logprob as fl


def test_rows_that_overlap_are_copied():
    """The fp32 and fp64 kernels take a row stride of at least a row: rows expanded from one, or
    cut from a longer one with overlap, are copied first."""
    row = torch.arange(12.0)
    for t in (row[:8].expand(5, 8), row.as_strided((3, 8), (2, 1)), row[:1].expand(4, 1), row[:8].reshape(8, 1).expand(8, 3)):
        got = fl._unit_stride(t)
        assert torch.equal(got, t) and got.stride(1) == 1 and got.stride(0) >= got.shape[1]
    padded = torch.zeros(4, 10)[:, :8]
    assert fl._unit_stride(padded) is padded and fl._unit_stride(row[None]).data_ptr() == row.data_ptr()
