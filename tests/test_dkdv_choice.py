"""The choice between the two dK/dV kernels at head dim 128 (CPU): launches timed
with both on an MI355X where one took at least 1.15 times the other's time take the
faster one."""

from __future__ import annotations

import pytest
import torch

from thundersync_amd import attention as att


def cohort(n, low, high, hq, hkv):
    lens = [low + (high - low) * i // (n - 1) for i in range(n)]
    return att._ragged_layout(lens, lens, hq, hkv)


def pack(n, low, high, prompt, hq, hkv):
    lens = [low + (high - low) * i // (n - 1) for i in range(n)]
    seg_q = tuple((sum(lens[:i]), m) for i, m in enumerate(lens))
    return att.AttnLayout(q_rows=sum(lens), hq=hq, hkv=hkv, source_rows=(prompt, *lens),
                          runs=tuple(att.Run(i, 0, m) for i, m in enumerate((prompt, *lens))), seg_q=seg_q,
                          seg_spans=tuple(((0, 0), (i + 1, prompt)) for i in range(n)))


CASES = [
    # layout, us dealt (48-key items), us key-split (64)
    (cohort(8, 512, 2048, 16, 8), 217.9, 182.7),
    (cohort(16, 256, 1024, 16, 8), 145.8, 100.9),
    (cohort(8, 128, 512, 16, 8), 36.0, 42.3),
    (cohort(4, 256, 1024, 16, 8), 41.3, 71.8),
    (cohort(16, 256, 1024, 24, 8), 190.2, 143.0),
    (cohort(8, 128, 512, 24, 8), 43.9, 57.9),
    (cohort(8, 512, 2048, 8, 8), 140.2, 102.9),
    (cohort(4, 256, 1024, 8, 8), 30.8, 41.3),
    (cohort(8, 1024, 4096, 32, 8), 1242.4, 1751.2),
    (att.chain_layout(256, [8192, 256], 40, 8), 175.1, 151.2),
    (att.chain_layout(256, [8192, 256], 24, 8), 130.0, 103.1),
    (att.chain_layout(64, [4096, 64], 32, 8), 42.9, 35.8),
    (att.chain_layout(1024, [4096, 1024], 32, 8), 205.3, 284.7),
    (att.chain_layout(256, [1024, 256], 32, 4), 38.3, 73.1),
    (pack(4, 32, 128, 4096, 24, 8), 80.6, 64.9),
    (pack(8, 64, 256, 1024, 8, 8), 39.3, 54.9),
    (pack(6, 200, 1500, 1500, 40, 8), 498.1, 812.9),
]


@pytest.mark.parametrize("case", range(len(CASES)))
def test_faster_kernel_is_chosen(case):
    layout, dealt, split = CASES[case]
    assert layout.call_kv_block(torch.device("cpu"), 128) == (48 if dealt < split else 64)
