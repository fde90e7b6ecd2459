"""One layout used on several streams: its tables are uploaded by the first call's
stream, and a call on another stream reads them after that."""

from __future__ import annotations

import pytest
import torch

from oracle import attention as ref
from thundersync_amd import _lib
from thundersync_amd import attention as hip


class _Blob(torch.Tensor):
    """A table tensor on the CPU that notes the streams it is recorded on."""

    log: list

    def record_stream(self, stream):
        self.log.append(("record", stream.cuda_stream))


@pytest.mark.parametrize("first, second", [(0, 7), (7, 0), (7, 9)])
def test_another_stream_waits_once(monkeypatch, first, second):
    """The tables' upload is what the other stream waits for, also when the
    default stream, whose handle is 0, is either of the two.  (CPU, streams and
    events that note what is asked of them; ExternalStream takes 0 for a stream
    of its own, as torch's does.)"""
    log, current, capturing = [], [first], [False]

    class Stream:
        def __init__(self, handle):
            self.cuda_stream = handle

        def wait_stream(self, other):
            self.wait_event(other.cuda_stream)

        def wait_event(self, event):
            log.append(("wait", self.cuda_stream, getattr(event, "stream", event)))

    class Event:
        def record(self, stream):
            self.stream = stream.cuda_stream

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
            blob = self.bytes.clone().as_subclass(_Blob)
            blob.log = log
            return blob

    monkeypatch.setattr(_lib, "current_stream", lambda device: current[0])
    monkeypatch.setattr(torch.cuda, "current_stream", lambda device=None: Stream(current[0]))
    monkeypatch.setattr(torch.cuda, "is_current_stream_capturing", lambda: capturing[0])
    monkeypatch.setattr(torch.cuda, "ExternalStream", lambda handle, device=None: Stream(handle or "another"))
    monkeypatch.setattr(torch.cuda, "Event", Event)
    lay = hip.chain_layout(70, [300], 4, 1)
    sources = [0x10000, 128, 128, 0x10000, 128, 128, 0, 0, 0, 0, 0, 0]
    monkeypatch.setattr(torch, "empty", lambda n, dtype=None, pin_memory=False: Host(n))
    upload = lambda: lay._upload(Device(), 64, sources)
    upload()
    upload()
    assert log == []
    current[0], capturing[0] = second, True
    upload()
    assert log == []
    capturing[0] = False
    upload()
    upload()
    assert log == [("wait", second, first), ("record", second)]


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
