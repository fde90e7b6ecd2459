"""One layout used on several streams: each reads the copy of its tables that it
uploaded itself."""

from __future__ import annotations

import pytest
import torch

from oracle import attention as ref
from thundersync_amd import _lib
from thundersync_amd import attention as hip


@pytest.mark.parametrize("first, second", [(0, 7), (7, 0), (7, 9)])
def test_each_stream_reads_its_own_upload(monkeypatch, first, second):
    """A stream's tables are a copy that this stream uploads, once, also when the
    default stream, whose handle is 0, is either of the two; a stream that
    captures adds no copy.  (CPU, copies that note the stream they are made on.)"""
    current, capturing, copies = [first], [False], []

    class Device:
        type, index = "cuda", 0

    class Host:
        """What a layout's build takes for pinned memory."""

        def __init__(self, n):
            self.bytes = torch.zeros(n, dtype=torch.uint8)

        def numpy(self):
            return self.bytes.numpy()

        def data_ptr(self):
            return self.bytes.data_ptr()

        def to(self, device, non_blocking):
            copies.append((current[0], self.bytes.numel(), self.bytes.clone()))
            return copies[-1][2]

    monkeypatch.setattr(_lib, "current_stream", lambda device: current[0])
    monkeypatch.setattr(torch.cuda, "is_current_stream_capturing", lambda: capturing[0])
    monkeypatch.setattr(torch, "empty", lambda n, dtype=None, pin_memory=False: Host(n))
    lay = hip.chain_layout(70, [300], 4, 1)
    sources = [0x10000, 128, 128, 0x10000, 128, 128, 0, 0, 0, 0, 0, 0]

    def upload(stream, capture=False):
        """A call's tables, and the streams that uploaded tables in it (a run table is smaller)."""
        current[0], capturing[0] = stream, capture
        copies.clear()
        tabs, _ = lay._upload(Device(), 64, sources)
        tables = [c for c in copies if c[1] > hip.RUN_DTYPE.itemsize]
        assert all(c[2] is tabs["blob"] for c in tables)
        return tabs, [c[0] for c in tables]

    one, by = upload(first)
    assert by == [first]
    assert upload(first) == (one, [])
    assert upload(second, capture=True) == (one, [])
    two, by = upload(second)
    assert by == [second] and two["blob"].data_ptr() != one["blob"].data_ptr()
    assert torch.equal(two["blob"], one["blob"])
    pointers = ("segs", "seg_spans", "run_visits_dev", "q_work", "kv_work", "dq_work", "span", "visit")
    shift = two["blob"].data_ptr() - one["blob"].data_ptr()
    assert [two[p] for p in pointers] == [one[p] and one[p] + shift for p in pointers]
    assert two["array_ptrs"] == one["array_ptrs"]
    assert upload(second) == (two, []) and upload(first) == (one, [])


@pytest.mark.gpu
@pytest.mark.parametrize("default_first", [False, True])
def test_two_streams(cuda, default_first):
    """The second stream's call is right though the first stream is still busy before the upload."""
    print(f"two streams, default stream first: {default_first}", flush=True)
    g = torch.Generator().manual_seed(0)
    q, do = (torch.randn(70, 4, 128, generator=g).bfloat16() for _ in range(2))
    k, v = (torch.randn(300, 1, 128, generator=g).bfloat16() for _ in range(2))
    want = ref.attention_with_grads(q, [k], [v], do, 0.1)
    q, do, k, v = (t.to(cuda) for t in (q, do, k, v))
    lay = hip.chain_layout(70, [300], 4, 1)
    busy = torch.randn(4096, 4096, device=cuda)
    torch.cuda.synchronize()
    results = []
    streams = [torch.cuda.Stream(), torch.cuda.Stream()]
    streams.insert(0 if default_first else 2, torch.cuda.current_stream())
    for stream in streams:
        with torch.cuda.stream(stream):
            if not results:
                for _ in range(20):
                    busy = busy @ busy * 1e-4
            leaves = [t.clone().requires_grad_() for t in (q, k, v)]
            out, _ = hip.attention(leaves[0], lay, [leaves[1]], [leaves[2]], 0.1)
            results.append((out, *torch.autograd.grad(out, leaves, do)))
    del lay
    torch.cuda.synchronize()
    for out, dq, dk, dv in results:
        for got, w in ((out, want[0]), (dq, want[1]), (dk, want[2][0]), (dv, want[3][0])):
            assert (got.detach().float().cpu() - w).abs().max().item() <= 2e-2 * max(1.0, w.abs().max().item())
