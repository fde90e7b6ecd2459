"""The native layout and run tables (CPU): the dQ pass's 64-row list, the
launch-order counts and the run table's rows recomputed item by item, and the
one-piece upload of a new layout with a call's run table."""

from __future__ import annotations

from pathlib import Path

import numpy as np
import pytest
import torch

from thundersync_amd import _lib
from thundersync_amd import attention as att

pytestmark = pytest.mark.skipif(_lib.library() is None, reason="libthundersync_hip.so not built")

CPU = torch.device("cpu")


def layouts():
    yield att.chain_layout(1, [1], 4, 1)
    yield att.chain_layout(65, [512, 17, 65], 32, 8)
    yield att._ragged_layout([5, 0, 130, 64], [9, 3, 130, 200], 8, 2)
    # a run nobody visits, a run two segments share, a head count without the 64-row list
    yield att.AttnLayout(q_rows=40, hq=10, hkv=2, source_rows=(100, 40), runs=(att.Run(0, 8, 50), att.Run(0, 60, 40),
                         att.Run(1, 0, 40)), seg_q=((0, 15), (15, 25)),
                         seg_spans=(((0, 0), (2, 50)), ((0, 0), (2, 50))))
    # re-read rows beyond half the shared cache: only long items run item-major
    yield att.chain_layout(9000, [40000, 9000], 32, 8)


@pytest.mark.parametrize("which", range(5))
def test_dq_list_counts_and_visits(which):
    lay = list(layouts())[which]
    *_, visit0, nvisit, q_long, kv_long, dq_work, dq_long = lay._host_tables()
    group = lay.hq // lay.hkv
    want = []
    if group % 4 == 0:
        for s, (_, n) in enumerate(lay.seg_q):
            want += [(lay.seg_kv[s] - n + min(q0 + 64, n), s, q0) for q0 in range(0, n, 64)]

    def band(cost):
        return int(np.floor(np.log(np.float64(max(cost, 1))) / np.log(1.0 + att.ORDER_BAND)))

    want.sort(key=lambda x: (-band(x[0]), x[1], x[2]))
    assert [tuple(x) for x in dq_work.tolist()] == [(s, q0) for _, s, q0 in want]
    users = [sum(1 for sp in lay.seg_spans for run, _ in sp if run == r) for r in range(len(lay.runs))]
    assert nvisit == users and visit0 == np.concatenate([[0], np.cumsum(users)])[:-1].tolist()

    def longs(costs, heads, reread):
        if reread <= 128 << 20:
            return len(costs)
        n, limit = 0, 0.25 * sum(costs) * heads / 256
        while n < len(costs) and costs[n] >= limit:
            n += 1
        return n

    kv_bytes = sum(r.length for r in lay.runs) * lay.hkv * 128 * 4
    assert dq_long == longs([c for c, _, _ in want], lay.hkv * (group // 4), kv_bytes)
    if kv_bytes <= 128 << 20:
        assert q_long == sum(-(-n // att.q_block_rows(lay.hq, lay.hkv)) for _, n in lay.seg_q)


def test_run_table_and_one_piece_upload():
    lay = list(layouts())[3]
    sources = [0x10000, 256, 128, 0x20000, 512, 64, 0, 0, 0, 0x30000, 256, 128,
               0x50000, 1024, 8, 0x60000, 2048, 16, 0x70000, 32, 8, 0, 0, 0]
    key = 64
    tabs, (ptr, host, (dev, _)) = lay._upload(CPU, key, sources)
    assert ptr == dev.data_ptr() + dev.numel() - host.size  # behind the tables, in the same buffer
    runs = host.view(att.RUN_DTYPE)
    again = lay._upload(CPU, key, sources)
    assert again[0] is tabs and again[1][0] != ptr and np.array_equal(again[1][1], host)
    for r, run in enumerate(lay.runs):
        x = sources[12 * run.source : 12 * run.source + 12]
        for j, name in enumerate(("k", "v", "dk", "dv")):
            address, row, head = x[3 * j : 3 * j + 3]
            assert runs[name][r] == (address + 2 * run.offset * row if address else 0)
            assert runs[f"{name}_row_stride"][r] == row and runs[f"{name}_head_stride"][r] == head
        assert runs["len"][r] == run.length
        assert (runs["visit0"][r], runs["nvisit"][r]) == (tabs["visit0"][r], tabs["nvisit"][r])


def test_arrays_outlive_the_call_that_reads_them(monkeypatch):
    """A layout's description may be made again by another thread while a call fills its
    run table: the arrays that the native code reads stay as long as it runs."""
    import gc
    import weakref

    lay = list(layouts())[3]
    tabs = lay.device_tables(CPU, 64)
    lib = _lib.require_library()

    class Library:
        @staticmethod
        def ts_attn_run_table(*args):
            arrays = [weakref.ref(a) for a in lay._desc["arrays"]]
            lay._desc = None
            gc.collect()
            assert all(a() is not None for a in arrays)
            return lib.ts_attn_run_table(*args)

        ts_hip_last_error = lib.ts_hip_last_error

    monkeypatch.setattr(_lib, "_LIB", Library())
    out = np.zeros(len(lay.runs), att.RUN_DTYPE)
    lay._fill_runs(tabs, [0x10000, 256, 128] * 8, out)
    assert out["len"].tolist() == [r.length for r in lay.runs]


def test_host_memory_is_an_error():
    """Tables that do not fit the host's memory are an error of the call, not the process's end."""
    import subprocess
    import sys

    code = """
import resource, ctypes, sys
from pathlib import Path

import numpy as np
from thundersync_amd import _lib, attention as att
from thundersync_amd._abi import AttnLayoutDesc, AttnLayoutSizes
lib = _lib.require_library()
lay = att.chain_layout(1 << 29, [1 << 29], 32, 8)
p = lay._description()["ptrs"]
desc = AttnLayoutDesc(lay.q_rows, 1, 32, 8, 1, 1, 48, 0, p[0], p[1], p[2], p[3])
sizes = AttnLayoutSizes()
assert lib.ts_attn_layout_tables(ctypes.byref(desc), None, 0, None, ctypes.byref(sizes)) == 0
run_visits, blob = np.zeros((1, 2), np.int32), np.zeros(sizes.bytes, np.uint8)  # pages come when they are written
used = int(open("/proc/self/statm").read().split()[0]) * resource.getpagesize()
resource.setrlimit(resource.RLIMIT_AS, (used + (64 << 20), resource.getrlimit(resource.RLIMIT_AS)[1]))
status = lib.ts_attn_layout_tables(ctypes.byref(desc), blob.ctypes.data, sizes.bytes, run_visits.ctypes.data, ctypes.byref(sizes))
sys.exit(0 if status != 0 else 3)
"""
    root = str(Path(__file__).resolve().parents[1])
    done = subprocess.run([sys.executable, "-c", code], capture_output=True, text=True, timeout=120, cwd=root)
    assert done.returncode == 0, (done.returncode, done.stderr[-400:])
