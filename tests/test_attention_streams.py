"""One layout used on several streams: its tables are uploaded by the first call's
stream, and a call on another stream reads them after that."""

from __future__ import annotations

import pytest
import torch

from oracle import attention as ref
from thundersync_amd import _lib
from thundersync_amd import attention as hip


def test_another_stream_waits_once(monkeypatch):
    """(CPU, streams that record what is asked of them.)"""
    log = []

    class Stream:
        def __init__(self, name):
            self.name, self.cuda_stream = name, name

        def wait_stream(self, other):
            log.append(("wait", self.name, other.name))

    class Blob:
        def record_stream(self, stream):
            log.append(("record", stream.name))

    first, second, capturing = Stream("first"), Stream("second"), [False]
    current = [first]
    monkeypatch.setattr(_lib, "current_stream", lambda device: current[0].cuda_stream)
    monkeypatch.setattr(torch.cuda, "current_stream", lambda device=None: current[0])
    monkeypatch.setattr(torch.cuda, "is_current_stream_capturing", lambda: capturing[0])
    monkeypatch.setattr(torch.cuda, "ExternalStream", lambda handle, device: {"first": first, "second": second}[handle])
    tabs = {"stream": "first", "streams": {"first"}, "blob": Blob()}
    device = torch.device("cuda:0")
    hip._order_after_upload(tabs, device)
    assert log == []
    current[0], capturing[0] = second, True
    hip._order_after_upload(tabs, device)
    assert log == []
    capturing[0] = False
    hip._order_after_upload(tabs, device)
    hip._order_after_upload(tabs, device)
    assert log == [("wait", "second", "first"), ("record", "second")]


@pytest.mark.gpu
def test_two_streams(cuda):
    """The second stream's call is right though the first stream is still busy before the upload."""
    print("two streams", flush=True)
    g = torch.Generator().manual_seed(0)
    q, do = (torch.randn(70, 4, 128, generator=g).bfloat16() for _ in range(2))
    k, v = (torch.randn(300, 1, 128, generator=g).bfloat16() for _ in range(2))
    want = ref.attention_with_grads(q, [k], [v], do, 0.1)
    q, do, k, v = (t.to(cuda) for t in (q, do, k, v))
    lay = hip.chain_layout(70, [300], 4, 1)
    busy = torch.randn(4096, 4096, device=cuda)
    torch.cuda.synchronize()
    results = []
    for stream in (torch.cuda.Stream(), torch.cuda.Stream(), torch.cuda.current_stream()):
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
