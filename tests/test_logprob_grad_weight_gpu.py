"""The weight gradient block by block: a first block that writes the fp32
accumulator, blocks that add to it and a last one that rounds, against the
plain add of every block to a zeroed accumulator and one cast -- the same fp32
sums in the same order, so the same bytes."""

from __future__ import annotations

import pytest
import torch

from thundersync_amd import _lib

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("vocab,dim,blocks", [
    (1, 8, [1]), (255, 264, [33]), (256, 256, [32, 32]), (257, 248, [64, 1]), (700, 520, [256, 300, 7]),
])
@pytest.mark.parametrize("dtype", [torch.bfloat16, torch.float16])
def test_blocks_equal_accumulate_and_cast(cuda, vocab, dim, blocks, dtype):
    print(f"grad_weight vocab={vocab} dim={dim} blocks={blocks} {dtype}", flush=True)
    lib = _lib.require_library()
    g = torch.Generator().manual_seed(vocab + dim)
    vp = (vocab + 7) // 8 * 8
    code = _lib.dtype_code(dtype)
    want = torch.zeros(vocab, dim, device=cuda)
    acc = torch.full((vocab, dim), float("nan"), device=cuda) if len(blocks) > 1 else None
    out = torch.full((vocab + 1, dim), 7.0, dtype=dtype, device=cuda)
    for i, rows in enumerate(blocks):
        dl = torch.randn(rows, vp, generator=g).to(dtype).to(cuda)
        h = torch.randn(rows, dim, generator=g).to(dtype).to(cuda)
        s = _lib.stream_of(h)
        _lib.check(lib.ts_logprob_grad_weight(dl.data_ptr(), vp, h.data_ptr(), dim, rows, dim, vocab, want.data_ptr(),
                                              dim, code, s), "add")
        last = i + 1 == len(blocks)
        _lib.check(lib.ts_logprob_grad_weight_block(dl.data_ptr(), vp, h.data_ptr(), dim, rows, dim, vocab,
                                                    _lib.ptr(acc), dim, int(i == 0), out.data_ptr() if last else None,
                                                    dim, code, s), "block")
    assert torch.equal(out[:vocab], want.to(dtype))
    assert bool((out[vocab] == 7.0).all())
