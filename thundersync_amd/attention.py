"""Forest / packed bottom-right-causal GQA attention on the gfx950 kernels.

One differentiable core op, :func:`attention`, serves every shape the
reference's streaming engine produces.  A call is described by an
:class:`AttnLayout`:

* **key sources** -- the K/V tensors the call reads, each ``[N, Hkv, D]``
  (a retained chunk, a pack's own K/V, a forest's whole K/V), read in place;
* **runs** -- contiguous row ranges of a source (a whole chunk, one forest
  node);
* **segments** -- blocks of query rows of the packed ``[R, Hq, D]`` query,
  each attending bottom-right-causally to the concatenation of its runs.

The layout is integer metadata only (no pointers), so one layout serves every
layer of a model call, as the reference's ``_PackLayout`` does
(src/thundersync/engine/streaming.py:1613-1698).  The pointer table is
rebuilt per call from the tensors themselves.

Reference entry points mirrored here (same argument meaning):

* :func:`causal_attention` -- the callable-backend form ``(query, ks, vs,
  scale) -> out`` that ``_causal_sdpa(..., backend=)`` dispatches to
  (engine/streaming.py:1094-1095) and ``grpo/attention.py:148-172`` provides;
* :class:`ChunkedCausalAttention` -- ``_ChunkedCausalSDPA.apply(query, scale,
  n_chunks, keep_state, backend, *ks, *vs)`` (engine/streaming.py:1314-1423);
* :class:`PackLayout` / :class:`PackedAttention` -- ``_PackedFlashSplit.apply(
  query, key, value, scale, layout, *ancestors)`` (engine/streaming.py:
  1613-1836), with ancestors in the reference's "last segment first" order;
* :func:`ragged_causal_attention` -- ``_ragged_causal_sdpa`` (:1165-1226),
  and :class:`RaggedAttention` -- ``_RaggedAttentionIndependentVJP``
  (:1253-1297);
* :func:`forest_attention` -- ``forest_attention(q, k, v, plan, *, scale)``
  (engine/attention.py:186-231);
* :func:`retained_chunk_layout` / :func:`retained_chunk_attention` -- every
  query chunk of a streamed pack over its retained per-chunk K/V in one
  launch, each chunk being the call ``_ChunkedCausalSDPA`` makes
  (engine/streaming.py:1314-1423).

Element types: bf16 and fp16 (Q, K, V of one call share one).  Head dims D:
any from 1 to 256, as the reference's flash paths take
(engine/streaming.py:532-548, :915-930).  The kernels are built for 32, 64,
96, 128, 192 and 256; any other D runs the next larger of them over Q, K and V
zero-padded to it (see :func:`kernel_head_dim`).  At head dims 128 and
256 the backward stores dS once in a workspace and forms dQ = dS K from it
(see ``DS_MAX_BYTES``).  There is no host path: CPU tensors, other dtypes or
head dims above 256 raise.
"""

from __future__ import annotations

import ctypes
import math
import os
import threading
from array import array
from collections.abc import Sequence
from dataclasses import dataclass, field
from itertools import chain
from typing import NamedTuple

import numpy as np
import torch

from . import _lib
from ._abi import REF_DTYPE, RUN_DTYPE, SEG_DTYPE, AttnLayoutDesc, AttnLayoutSizes, AttnProblem, AttnRows
from .dispatch import HIP_BACKWARD_PATH, HIP_PATH, count_attention_path
from .operator_profiling import operator_range

HEAD_DIMS = (32, 64, 96, 128, 192, 256)  # the head dims the kernels are built for
MAX_HEAD_DIM = 256
HEAD_DIM = 128  # the head dim the tuned kernels take; also the launch-order estimate's row width
ELEMENT_DTYPES = (torch.bfloat16, torch.float16)


def heads_per_block(group: int) -> int:
    """Query heads per forward/dQ work-group (mirror of ts_attn_heads_per_block)."""
    if group % 4 == 0:
        return 4
    if group % 2 == 0:
        return 2
    return 1


def q_block_rows(hq: int, hkv: int) -> int:
    """Query rows per forward/dQ work item (mirror of ts_attn_q_block)."""
    return 32 * 4 // heads_per_block(hq // hkv)


def kv_block_keys(hq: int, hkv: int, head_dim: int = HEAD_DIM) -> int:
    """Keys per dK/dV work-group (mirror of ts_attn_kv_block): 64 at head dim
    256 and for GQA groups that are not a multiple of 4, else 48."""
    return 48 if (hq // hkv) % 4 == 0 and head_dim != 256 else 64


# At head dim 256 the 64-key dK/dV work items run two work-groups per CU
# (two waves of 32 keys each); a launch with fewer of them than that fills
# (512) leaves CUs half used, and the 48-key items of the key-split kernel
# (one work-group per CU, four waves of 16 keys) balance better: the branch
# shape at 16/2 heads (384 items of 64 keys) 7.06 ms against 6.54.
DKDV256_MIN_ITEMS = 512


# At head dim 128, 48-key dK/dV items run the kernel whose waves take steps
# (a query head, 32 rows) of their own, 64-key items the key-split kernel, whose
# waves take 16 keys each of every step.  The first does each step in fewer LDS
# reads and without a barrier, the second starts and ends cheaper (16 keys'
# operands to load, no partials to sum over the waves) and holds two
# work-groups a CU.  So the first pays where items have many steps, the second
# where there are many items of few.  A launch takes about
#     start + round * rounds + step * max(tail * longest item's steps, steps a slot)
# us, slots being the work-groups the device holds at once and rounds the items
# over them: fitted to 266 launches (one sequence over a context, cohorts, packs; 16
# to 9000 rows over up to 14000 keys) at head counts from 32/4 to 8/8, where the
# choice costs 0.4 % on average and at most 13 % (24/8 heads, 8 sequences of 512 to
# 2048 rows: 290 us dealt, 258 split; outside them 133 rows over 1605 keys at 40/8,
# just past one round of dealt items: 50 and 35).  By the average steps of an item
# alone it cost 3.6 % and up to 79 %: dealt against split 146 / 101 us for 16
# sequences of 256 to 1024 rows at 16/8, 130 / 103 for 256 rows over 8448 keys at
# 24/8, 31 / 41 for 4 sequences of 256 to 1024 rows at 8/8.
def _dealt_is_faster(items48: int, items64: int, group: int, mean: float, most: int) -> bool:
    """Whether 48-key items are estimated to end sooner than 64-key ones, given
    the items of either size and the query rows that an item sees, on average and
    at most.  Dealt out: start 4, round 12, step 0.46 us, tail 0.7 over 256 slots;
    key-split: 10, none, 1.8, 0.55 over 512."""
    dealt, split = items48 / 256, items64 / 512  # rounds
    steps = group / 32  # of a row
    return (4.0 + 12.0 * max(dealt, 1.0) + 0.46 * steps * max(0.7 * most, mean * dealt)
            < 10.0 + 1.8 * steps * max(0.55 * most, mean * split))


# ---------------------------------------------------------------------------
# layout
# ---------------------------------------------------------------------------
class Run(NamedTuple):
    source: int  # index into the call's key sources
    offset: int  # first row within the source
    length: int


@dataclass(eq=False)
class AttnLayout:
    """Integer description of one attention call (see the module docstring)."""

    q_rows: int
    hq: int
    hkv: int
    source_rows: tuple[int, ...]
    runs: tuple[Run, ...]
    seg_q: tuple[tuple[int, int], ...]  # (q_row0, q_len) per segment
    seg_spans: tuple[tuple[tuple[int, int], ...], ...]  # per segment: (run, kpos)
    seg_kv: tuple[int, ...] = field(init=False)
    _tables: dict = field(default_factory=dict, init=False, repr=False)
    _lock: threading.Lock = field(default_factory=threading.Lock, init=False, repr=False)
    _desc: dict | None = field(default=None, init=False, repr=False)

    def __post_init__(self):
        if self.hq <= 0 or self.hkv <= 0 or self.hq % self.hkv:
            raise ValueError(f"query heads {self.hq} are not a multiple of KV heads {self.hkv}")
        runs, sources = self.runs, self.source_rows
        n_runs, n_sources = len(runs), len(sources)
        kv = []
        for s, spans in enumerate(self.seg_spans):
            pos = 0
            for run, kpos in spans:
                if not 0 <= run < n_runs:
                    raise ValueError(f"segment {s} names run {run} of {n_runs}")
                if kpos != pos:
                    raise ValueError(f"segment {s}: spans must tile its keys in order (kpos {kpos} != {pos})")
                pos += runs[run][2]
            kv.append(pos)
        self.seg_kv = tuple(kv)
        if len(self.seg_q) != len(self.seg_spans):
            raise ValueError("one span list per segment")
        for s, (row0, length) in enumerate(self.seg_q):
            if length < 0 or row0 < 0 or row0 + length > self.q_rows:
                raise ValueError(f"segment {s} rows [{row0}, {row0 + length}) outside [0, {self.q_rows})")
            if length > 0 and kv[s] < length:
                raise ValueError(
                    f"segment {s} has {length} query rows but only {kv[s]} keys; "
                    "bottom-right causal attention needs kv_len >= q_len"
                )
        for r, (source, offset, length) in enumerate(runs):
            if not 0 <= source < n_sources:
                raise ValueError(f"run {r} names source {source}")
            if length <= 0 or offset < 0 or offset + length > sources[source]:
                raise ValueError(f"run {r} rows outside its source")
        # the backward writes each run's dK/dV through its own rows, without
        # atomics: two runs may not share a row of a source
        if len({r[0] for r in runs}) != n_runs:
            by_source: dict[int, list[tuple[int, int, int]]] = {}
            for r, (source, offset, length) in enumerate(runs):
                by_source.setdefault(source, []).append((offset, offset + length, r))
            for source, spans in by_source.items():
                spans.sort()
                for (a0, a1, ra), (b0, _b1, rb) in zip(spans, spans[1:]):
                    if b0 < a1:
                        raise ValueError(f"runs {ra} and {rb} overlap in source {source} (rows {b0}..{a1 - 1})")
        if max([*kv, 0]) >= 2**31 or self.q_rows >= 2**40:
            raise ValueError("attention problem too large")

    # -- tables -------------------------------------------------------------
    def _description(self) -> dict:
        """The layout as the native table builder takes it (host arrays and
        their addresses), made once."""
        d = self._desc
        if d is None:
            span0, at = array("q", (0,)), 0
            for spans in self.seg_spans:
                at += len(spans)
                span0.append(at)
            spans = array("i", chain.from_iterable(chain.from_iterable(self.seg_spans)))
            arrays = (array("q", chain.from_iterable(self.seg_q)), span0, spans, array("i", (r[2] for r in self.runs)),
                      array("i", (r[0] for r in self.runs)), array("q", (r[1] for r in self.runs)))
            # visited runs: query rows of the segments that read them
            if len(self.seg_q) == 1:
                users = dict.fromkeys(spans[::2], self.seg_q[0][1])
            else:
                users = {}
                for (_, n), seg in zip(self.seg_q, self.seg_spans):
                    for r, _ in seg:
                        users[r] = users.get(r, 0) + n
            # rows of each source that a visited run covers (runs do not overlap)
            covered, key_rows, items48, items64 = [0] * len(self.source_rows), 0, 0, 0
            for r in users:
                source, _, length = self.runs[r]
                covered[source] += length
                key_rows += length
                items48 += (length + 47) // 48
                items64 += (length + 63) // 64
            d = {
                "arrays": arrays,
                "ptrs": tuple(a.buffer_info()[0] if len(a) else None for a in arrays),
                "n_spans": at,
                # dK/dV items of one KV head, by their size
                "items64": items64,
                # sources with rows that no visited run covers: their gradients are filled with zeros first
                "uncovered": [i for i, n in enumerate(self.source_rows) if covered[i] != n],
                "kv_block128": 48 if _dealt_is_faster(
                    items48 * self.hkv, items64 * self.hkv, self.hq // self.hkv,
                    self.visible_pairs() / max(key_rows, 1), max(users.values(), default=0)) else 64,
                "max_keys": max((kv for kv, (_, n) in zip(self.seg_kv, self.seg_q) if n), default=0),
                "all_rows": sum(n for _, n in self.seg_q) == self.q_rows,
            }
            self._desc = d
        return d

    def _build(self, kvb: int, alloc, extra: int = 0):
        """(sizes, buffer from ``alloc(bytes)``, its numpy view, run_visits): the
        layout's tables at the start of the buffer, ``extra`` bytes after them."""
        lib = _lib.require_library()
        d = self._description()
        p = d["ptrs"]
        desc = AttnLayoutDesc(self.q_rows, d["n_spans"], self.hq, self.hkv, len(self.seg_q), len(self.runs), kvb, 0,
                              p[0], p[1], p[2], p[3])
        sizes = AttnLayoutSizes()
        _lib.check(lib.ts_attn_layout_tables(ctypes.byref(desc), None, 0, None, ctypes.byref(sizes)),
                   "ts_attn_layout_tables")
        buf = alloc(sizes.bytes + extra)
        view = buf if isinstance(buf, np.ndarray) else buf.numpy()
        run_visits = np.zeros((max(len(self.runs), 1), 2), np.int32)
        _lib.check(lib.ts_attn_layout_tables(ctypes.byref(desc), view.ctypes.data, sizes.bytes,
                                             run_visits.ctypes.data, ctypes.byref(sizes)), "ts_attn_layout_tables")
        return sizes, buf, view, run_visits

    def _views(self, sizes: AttnLayoutSizes, view: np.ndarray):
        """(segs, spans, visits, q_work, kv_work, dq_work) as views of a table buffer."""
        n = self._description()["n_spans"]

        def part(offset, count, dtype):
            return view[offset : offset + count * dtype.itemsize].view(dtype)

        pair = np.dtype(np.int32)
        return (part(sizes.segs, len(self.seg_q), SEG_DTYPE), part(sizes.spans, n, REF_DTYPE),
                part(sizes.visits, n, REF_DTYPE), part(sizes.q_work, 2 * sizes.n_q_work, pair).reshape(-1, 2),
                part(sizes.kv_work, 2 * sizes.n_kv_work, pair).reshape(-1, 2),
                part(sizes.dq_work, 2 * sizes.n_dq_work, pair).reshape(-1, 2))

    def _host_tables(self, kvb: int | None = None):
        kvb = kv_block_keys(self.hq, self.hkv) if kvb is None else kvb
        sizes, _, view, run_visits = self._build(kvb, lambda n: np.zeros(n, np.uint8))
        segs, spans, visits, q_work, kv_work, dq_work = self._views(sizes, view)
        rv = run_visits[: len(self.runs)]
        return (segs, spans, visits, q_work, kv_work, rv[:, 0].tolist(), rv[:, 1].tolist(),
                int(sizes.n_q_long), int(sizes.n_kv_long), dq_work, int(sizes.n_dq_long))

    def _fill_runs(self, tabs: dict, sources: Sequence[int], out: np.ndarray) -> None:
        """One call's run table into ``out`` (``sources``: ts_attn_run_table's)."""
        d = self._description()  # held: `_desc` may be another thread's by the time the native code reads the arrays
        p = d["ptrs"]
        src = array("q", sources)
        _lib.check(
            _lib.require_library().ts_attn_run_table(
                len(self.runs), p[3], p[4], p[5], tabs["run_visits_ptr"], len(self.source_rows),
                src.buffer_info()[0] if len(src) else None, out.ctypes.data if len(self.runs) else None),
            "ts_attn_run_table",
        )

    def _upload(self, device: torch.device, kvb: int, sources: Sequence[int] | None):
        """(tables, run table): the layout's tables on ``device``, built once per
        device and dK/dV item size and uploaded once per stream, and, with
        ``sources``, one call's run table as (device address, host bytes, tensors
        to keep).  Both go through pinned memory without blocking, in one piece
        when the layout is new.  A stream reads the copy that it uploaded itself,
        so no stream waits for another and the copy's memory is its own; a stream
        that is capturing takes another's, if there is one, without a copy in the
        graph.  (With an event recorded behind the upload for other streams to
        wait on, a 48-row turn took 121 us; so 111 to 113.)"""
        stream = _lib.current_stream(device) if device.type == "cuda" else 0
        at = (device.type, device.index, kvb)
        key = (*at, stream)
        run_bytes = len(self.runs) * RUN_DTYPE.itemsize if sources is not None else 0

        def alloc(n):
            return torch.empty(max(n, 16), dtype=torch.uint8, pin_memory=device.type == "cuda")

        tabs = self._tables.get(key)
        if tabs is None:
            with self._lock:
                tabs = self._tables.get(key)
                first = None if tabs else next((t for k, t in self._tables.items() if k[:3] == at), None)
                if first is not None:
                    tabs = first
                    if not torch.cuda.is_current_stream_capturing():
                        tabs = self._tables[key] = self._on_device(first, first["host"], first["sizes"], device)
                elif tabs is None:
                    sizes, host, view, run_visits = self._build(kvb, alloc, run_bytes)
                    segs, spans, visits, q_work, kv_work, _ = self._views(sizes, view)
                    n = self._description()["n_spans"]
                    tabs = {
                        "run_visits": run_visits,
                        "run_visits_ptr": run_visits.ctypes.data,
                        "arrays": (segs, spans, visits, q_work, kv_work),
                        "array_ptrs": tuple(a.ctypes.data if a.size else None
                                            for a in (segs, spans, visits, q_work, kv_work)),
                        "visit0": run_visits[: len(self.runs), 0].tolist(),
                        "nvisit": run_visits[: len(self.runs), 1].tolist(),
                        "n_q_work": int(sizes.n_q_work), "n_kv_work": int(sizes.n_kv_work),
                        "n_dq_work": int(sizes.n_dq_work), "n_q_long": int(sizes.n_q_long),
                        "n_kv_long": int(sizes.n_kv_long), "n_dq_long": int(sizes.n_dq_long),
                        "head": int(sizes.ds_head),
                        "span_ds": view[sizes.span_ds : sizes.span_ds + 8 * n].view(np.int64),
                        "visit_ds": view[sizes.visit_ds : sizes.visit_ds + 8 * n].view(np.int64),
                    }
                    if run_bytes:
                        self._fill_runs(tabs, sources, view[sizes.bytes :])
                    tabs = self._tables[key] = self._on_device(tabs, host, sizes, device)
                    if sources is not None:
                        dev = tabs["blob"]
                        return tabs, (dev.data_ptr() + sizes.bytes,
                                      view[sizes.bytes : sizes.bytes + run_bytes], (dev, host))
        if sources is None:
            return tabs, None
        host = alloc(run_bytes)
        view = host.numpy()
        self._fill_runs(tabs, sources, view)
        dev = host.to(device, non_blocking=True)
        return tabs, (dev.data_ptr(), view[:run_bytes], (dev, host))

    @staticmethod
    def _on_device(tabs: dict, host: torch.Tensor, sizes: AttnLayoutSizes, device: torch.device) -> dict:
        """The tables with a copy of ``host`` that the current stream uploads."""
        dev = host.to(device, non_blocking=True)
        base = dev.data_ptr()
        return dict(
            tabs, blob=dev, host=host, sizes=sizes, segs=base + sizes.segs, seg_spans=base + sizes.spans,
            run_visits_dev=base + sizes.visits, q_work=base + sizes.q_work, kv_work=base + sizes.kv_work,
            dq_work=base + sizes.dq_work if sizes.n_dq_work else None,
            span=base + sizes.span_ds, visit=base + sizes.visit_ds,
        )

    def device_tables(self, device: torch.device, kv_block: int | None = None):
        """The layout's integer tables on ``device``, uploaded once per stream
        and dK/dV item size (pinned, non-blocking); `kv_block` None: the
        head-dim-128 size."""
        kvb = kv_block_keys(self.hq, self.hkv) if kv_block is None else int(kv_block)
        return self._upload(device, kvb, None)[0]

    def ds_tables(self, device: torch.device, kv_block: int | None = None) -> dict:
        """The dS route's workspace layout: elements per head ("head") and the
        per-span / per-visit element offsets on the device ("span", "visit") and
        the host ("span_ds", "visit_ds"); part of the layout's tables."""
        return self.device_tables(device, kv_block)

    def kv_block_for(self, device, head_dim: int) -> int:
        """Keys per dK/dV work item at `head_dim`: ts_attn_kv_block's, except
        at head dim 256 when the 64-key items of the visited runs, over all
        KV heads, are fewer than DKDV256_MIN_ITEMS: then 48 (the key-split
        kernel)."""
        kvb = kv_block_keys(self.hq, self.hkv, head_dim)
        if head_dim == 256:
            if self._description()["items64"] * self.hkv < DKDV256_MIN_ITEMS:
                kvb = 48
        return kvb

    def call_kv_block(self, device, head_dim: int) -> int:
        """Keys per dK/dV work item of this package's own calls: kv_block_for's,
        except that at head dim 128 every GQA group takes either kernel, whichever
        is estimated to end sooner (_dealt_is_faster), and at the head dims that only the
        key-split kernel takes, whose four waves hold 16 keys each, every group has
        64."""
        if head_dim == 256:
            return self.kv_block_for(device, head_dim)
        if head_dim != HEAD_DIM:
            return 64
        return self._description()["kv_block128"]

    def problem(self, device, runs_ptr: int, scale: float, dtype: torch.dtype = torch.bfloat16,
                head_dim: int = HEAD_DIM, kv_block: int | None = None, tables: dict | None = None) -> AttnProblem:
        kvb = self.kv_block_for(device, int(head_dim)) if kv_block is None else kv_block
        t = tables or self.device_tables(device, kvb)
        return AttnProblem(
            t["segs"], t["seg_spans"], runs_ptr, t["run_visits_dev"], t["q_work"], t["kv_work"],
            t["n_q_work"], t["n_kv_work"], len(self.seg_q), len(self.runs), self.hq, self.hkv,
            int(head_dim), float(scale), q_block_rows(self.hq, self.hkv), kvb, self.q_rows,
            t["n_q_long"], t["n_kv_long"], _lib.dtype_code(dtype),
        )

    # -- reference diagnostics ---------------------------------------------
    def visible_pairs(self) -> int:
        """Exactly visible (query, key) pairs, per head: sum over segments."""
        total = 0
        for (_, t), s in zip(self.seg_q, self.seg_kv):
            total += t * (s - t) + t * (t + 1) // 2
        return total


# Work items are launched in bands of costs within ORDER_BAND of each other
# (geometric), longest band first, and within a band by run (dK/dV) or
# segment (forward, dQ) and position: neighbours in the list, which the
# launch order places on one XCD together, then read the same rows and share
# its L2, while the longest-first order that keeps the end of the launch
# short changes by at most ORDER_BAND.  (C4: dK/dV 34.3 -> 32.4 ms, forward
# 11.85 -> 11.62 ms, dQ 10.7 -> 10.0 ms; C2 within noise.)
#
# The first n_*_long items of a list run item-major at the head of the launch:
# when the rows the work-groups re-read (all heads) fit in half the shared
# last-level cache (256 MB), every item does -- each XCD then serves fixed heads
# and keeps their rows in its L2 while the shared cache holds the rest.
# Otherwise only the items long enough to stretch the end of the launch when
# started late -- a quarter or more of a slot's average share of the whole
# launch -- and the rest run head by head, all XCDs streaming one head's rows
# through the shared cache.  ts_attn_layout_tables builds the lists, by its own
# copy of this constant (kOrderBand, attention_tables.hip); this one is for readers
# of the lists.
ORDER_BAND = 0.05


def _check_rows_tensor(t: torch.Tensor, name: str, heads: int, head_dim: int, max_row_stride: int = 1 << 24) -> None:
    if t.dim() != 3 or t.shape[1] != heads or t.shape[2] != head_dim:
        raise ValueError(f"{name} must be [rows, {heads}, {head_dim}], got {tuple(t.shape)}")
    if t.stride(2) != 1 or t.stride(0) % 8 or t.stride(1) % 8 or t.data_ptr() % 16:
        raise ValueError(f"{name} needs a contiguous head dim, 16-byte alignment and 8-element strides")
    if t.stride(0) >= max_row_stride:
        # the kernels address a tile's rows with 32-bit byte offsets
        raise ValueError(f"{name} row stride {t.stride(0)} must be below {max_row_stride} elements")


def _rows(t: torch.Tensor) -> AttnRows:
    return AttnRows(t.data_ptr(), t.stride(0), t.stride(1))


def check_tables(layout: AttnLayout, problem: AttnProblem, run_table: np.ndarray | torch.Tensor,
                 device: torch.device, tables: dict | None = None) -> None:
    """Check the layout's tables for ``device`` and one call's run table on the
    host (ts_attn_check_tables) before the kernels read their device copies:
    spans tile every segment's keys, every visit is a span of its segment,
    the work lists hold every row and key block once, K/V/dK/dV addresses are
    aligned.  Raises RuntimeError naming the first inconsistency."""
    tabs = tables or layout.device_tables(device, problem.kv_block)
    runs = run_table.numpy() if isinstance(run_table, torch.Tensor) else run_table
    runs = np.ascontiguousarray(runs).view(np.uint8)
    if runs.size != len(layout.runs) * RUN_DTYPE.itemsize:
        raise ValueError(f"run table holds {runs.size} bytes, expected {len(layout.runs)} runs")
    segs, spans, visits, q_work, kv_work = tabs["array_ptrs"]
    n_spans = layout._description()["n_spans"]
    lib = _lib.require_library()
    _lib.check(
        lib.ts_attn_check_tables(ctypes.byref(problem), segs, spans, n_spans, runs.ctypes.data if runs.size else None,
                                 visits, n_spans, q_work, kv_work),
        lambda: f"attention tables (rows={layout.q_rows}, segments={len(layout.seg_q)}, runs={len(layout.runs)})",
    )


def _validate_call(layout: AttnLayout, query: torch.Tensor, keys, values) -> None:
    if not query.is_cuda:
        raise RuntimeError("thundersync_amd attention runs on the GPU only; got a CPU tensor")
    if query.dtype not in ELEMENT_DTYPES:
        raise TypeError(f"thundersync_amd attention takes bf16 or fp16, got {query.dtype}")
    head_dim = query.shape[-1] if query.dim() == 3 else -1
    if head_dim not in HEAD_DIMS:
        raise ValueError(f"thundersync_amd attention takes head dims 1..{MAX_HEAD_DIM} (kernels at {HEAD_DIMS}), "
                         f"got query {tuple(query.shape)}")
    _check_rows_tensor(query, "query", layout.hq, head_dim)
    if query.shape[0] != layout.q_rows:
        raise ValueError(f"query has {query.shape[0]} rows, layout {layout.q_rows}")
    if len(keys) != len(layout.source_rows) or len(values) != len(layout.source_rows):
        raise ValueError("one K and one V tensor per key source")
    for i, (k, v) in enumerate(zip(keys, values)):
        for name, t in (("key", k), ("value", v)):
            if t.device != query.device or t.dtype != query.dtype:
                raise ValueError(f"{name} source {i} must be {query.dtype} on {query.device}")
            _check_rows_tensor(t, f"{name} source {i}", layout.hkv, head_dim)
            if t.shape[0] != layout.source_rows[i]:
                raise ValueError(f"{name} source {i} has {t.shape[0]} rows, layout {layout.source_rows[i]}")


# dS workspace (bytes) the backward may allocate for the dS route (dK/dV
# kernels store dS, dQ = dS K from it; about 2 bytes per visible pair and
# head): up to DS_MAX_BYTES, and a workspace above it when it fits in
# DS_FREE_FRACTION of the memory the device can still supply (an MI355X holds
# 288 GB; the reference's 16-trajectory retained-chunk pack needs ~52 GB);
# never more than DS_AVAILABLE_FRACTION of that memory, so a device that is
# nearly full takes the route over fewer KV heads, or not at all, instead of
# failing inside the backward.  The memory the device can supply is its free
# memory plus what torch's allocator holds unused.  A problem above the cap
# runs the route over groups of KV heads, as many per call as fit (KV heads
# are independent: their query heads, dS and gradients do not mix, and the
# grouped calls give the one-call gradients bit for bit); one whose single KV
# head does not fit, one whose workspace allocation fails all the same, or
# any under THUNDERSYNC_ATTN_DS=off, runs the route that recomputes S and dP
# in the dQ kernel.
DS_MAX_BYTES = 16 << 30
DS_FREE_FRACTION = 0.25
DS_AVAILABLE_FRACTION = 0.5
DS_ENV = "THUNDERSYNC_ATTN_DS"


def _device_free_bytes(device: torch.device) -> int:
    """Memory `device` can still supply in bytes: free device memory plus the
    allocator's reserved but unallocated bytes (0 for a host device)."""
    if device.type != "cuda":
        return 0
    free, _total = torch.cuda.mem_get_info(device)
    return int(free) + _device_cached_bytes(device)


def _device_cached_bytes(device: torch.device) -> int:
    """Bytes torch's allocator holds on `device` unallocated (0 for a host device)."""
    if device.type != "cuda":
        return 0
    stats = torch.cuda.memory_stats_as_nested_dict(device)
    if not stats:
        return 0
    return max(int(stats["reserved_bytes"]["all"]["current"]) - int(stats["allocated_bytes"]["all"]["current"]), 0)


def _ds_route(layout: AttnLayout, query: torch.Tensor, lib):
    """(workspace tables, KV heads per call) when this backward takes the dS
    route, else None."""
    if os.environ.get(DS_ENV, "auto").strip().lower() == "off" or DS_MAX_BYTES <= 0:
        return None
    group = layout.hq // layout.hkv
    if not lib.ts_attn_ds_route(query.shape[2], group):
        return None
    tabs = layout.ds_tables(query.device, layout.call_kv_block(query.device, query.shape[2]))
    # a call over n KV heads needs (n * group * head + 512) elements: every
    # query head's part, then the sink block
    per_kv_head = group * max(tabs["head"], 1)
    need = (layout.hkv * per_kv_head + 512) * 2
    if need <= DS_MAX_BYTES and need <= int(_device_cached_bytes(query.device) * DS_AVAILABLE_FRACTION):
        return tabs, layout.hkv  # the allocator's unused memory alone is enough: the device need not be asked
    available = _device_free_bytes(query.device)
    cap = DS_MAX_BYTES
    if (layout.hkv * per_kv_head + 512) * 2 > cap and DS_FREE_FRACTION > 0:
        cap = max(cap, int(available * DS_FREE_FRACTION))
    cap = min(cap, int(available * DS_AVAILABLE_FRACTION))
    kv_heads = min(layout.hkv, (cap // 2 - 512) // per_kv_head)
    if kv_heads < 1:
        return None
    return tabs, kv_heads


def _head_rows(rows: AttnRows, first_head: int) -> AttnRows:
    """A rows view that starts at head `first_head` (2-byte elements)."""
    return AttnRows(rows.ptr + first_head * rows.head_stride * 2, rows.row_stride, rows.head_stride)


def _head_runs(host: np.ndarray, first_kv_head: int, device) -> tuple[torch.Tensor, torch.Tensor]:
    """A copy of a run table whose K/V/dK/dV addresses start at KV head `first_kv_head`."""
    table = host.view(RUN_DTYPE).copy()
    for name in ("k", "v", "dk", "dv"):
        live = table[name] != 0
        table[name][live] += (first_kv_head * table[f"{name}_head_stride"][live] * 2).astype(np.uint64)
    sub = torch.from_numpy(table.view(np.uint8)).pin_memory() if device.type == "cuda" else torch.from_numpy(
        table.view(np.uint8))
    return sub.to(device, non_blocking=True), sub


def _gather(layout: AttnLayout, query: torch.Tensor, keys, values) -> list[int]:
    """Validate a call's tensors and list its K/V sources for the run table
    (12 numbers a source: k, v, dk, dv as address, row stride, head stride; the
    gradients zero).  Raises as :func:`_validate_call`, which the tests of one
    look per tensor below stand for."""
    if not query.is_cuda or query.dim() != 3 or len(keys) != len(layout.source_rows) or len(values) != len(keys):
        _validate_call(layout, query, keys, values)
    dtype, device, hkv, d = query.dtype, query.get_device(), layout.hkv, query.shape[2]
    qs = query.stride()
    plain = (dtype in ELEMENT_DTYPES and d in HEAD_DIMS and query.shape == (layout.q_rows, layout.hq, d)
             and qs[2] == 1 and not (qs[0] | qs[1]) & 7 and not query.data_ptr() & 15 and qs[0] < 1 << 24)
    out: list[int] = []
    for n, k, v in zip(layout.source_rows, keys, values):
        ks, vs, kp, vp = k.stride(), v.stride(), k.data_ptr(), v.data_ptr()
        shape = (n, hkv, d)
        if not (plain and k.dtype is dtype and v.dtype is dtype and k.shape == shape and v.shape == shape
                and k.get_device() == device and v.get_device() == device and ks[2] == 1 and vs[2] == 1
                and not (ks[0] | ks[1] | vs[0] | vs[1]) & 7 and not (kp | vp) & 15
                and ks[0] < 1 << 24 and vs[0] < 1 << 24):
            _validate_call(layout, query, keys, values)
        out += (kp, ks[0], ks[1], vp, vs[0], vs[1], 0, 0, 0, 0, 0, 0)
    if not plain:
        _validate_call(layout, query, keys, values)
    return out


def _parts_workspace(nbytes: int, device) -> torch.Tensor | None:
    """Memory for the partial sums of work items cut into parts, None where the
    device has none left (the items then stay whole)."""
    try:
        return torch.empty(nbytes, dtype=torch.uint8, device=device)
    except torch.cuda.OutOfMemoryError:
        return None


def _attention_forward(query: torch.Tensor, layout: AttnLayout, scale: float, keys, values):
    """(out, lse, tensors to keep while the launch reads them)."""
    sources = _gather(layout, query, keys, values)
    lib = _lib.require_library()
    device = query.device
    out = torch.empty(query.shape, dtype=query.dtype, device=device)
    lse = torch.empty(layout.hq, max(layout.q_rows, 1), dtype=torch.float32, device=device)
    kvb = layout.call_kv_block(device, query.shape[2])
    tabs, (runs, host, keep) = layout._upload(device, kvb, sources)
    problem = layout.problem(device, runs, scale, query.dtype, query.shape[2], kvb, tabs)
    check_tables(layout, problem, host, device, tabs)
    # few work items over many keys: each item's keys in several work-groups
    at = ctypes.byref(problem)
    parts = lib.ts_attn_fwd_parts(at, layout._description()["max_keys"])
    work = None
    if parts > 1:
        work = _parts_workspace(lib.ts_attn_fwd_parts_workspace(at, parts), device)
        parts = parts if work is not None else 1
    with operator_range("hip_attention_forward", rows=layout.q_rows, segments=len(layout.seg_q)):
        _lib.check(
            lib.ts_attn_fwd_split(at, _rows(query), _rows(out), lse.data_ptr(), lse.shape[1],
                                  parts, _lib.ptr(work), 0 if work is None else work.numel(),
                                  _lib.stream_of(query)),
            lambda: f"ts_attn_fwd(rows={layout.q_rows}, hq={layout.hq}, hkv={layout.hkv})",
        )
    count_attention_path(HIP_PATH)
    return out, lse, keep


def _attention_backward(query, out, lse, dout, layout: AttnLayout, scale: float, keys, values):
    """(dq, dkeys, dvalues, tensors to keep while the launches read them)."""
    lib = _lib.require_library()
    device = query.device
    if dout.stride(2) != 1 or dout.stride(0) % 8 or dout.stride(1) % 8:
        dout = dout.contiguous()
    # dQ in the query's own layout where it is dense (a [1, Hq, T, D] query
    # seen as rows gets its gradient without a copy into that layout)
    dq = torch.empty_like(query)
    if dq.stride(2) != 1 or dq.stride(0) % 8 or dq.stride(1) % 8:
        dq = torch.empty(query.shape, dtype=query.dtype, device=device)
    desc = layout._description()
    if not desc["all_rows"]:
        dq.zero_()
    dkeys = [torch.empty(k.shape, dtype=k.dtype, device=device) for k in keys]
    dvalues = [torch.empty(v.shape, dtype=v.dtype, device=device) for v in values]
    # rows of a source that no run covers, or runs nobody reads, get zeros
    for i in desc["uncovered"]:
        dkeys[i].zero_()
        dvalues[i].zero_()
    sources = _gather(layout, query, keys, values)
    d = query.shape[2]
    for i, (dk, dv) in enumerate(zip(dkeys, dvalues)):  # contiguous [rows, Hkv, D]
        sources[12 * i + 6 : 12 * i + 12] = (dk.data_ptr(), layout.hkv * d, d, dv.data_ptr(), layout.hkv * d, d)
    kvb = layout.call_kv_block(device, d)
    tabs, (runs, host, keep_runs) = layout._upload(device, kvb, sources)
    rowstats = torch.empty(layout.hq, max(layout.q_rows, 1), 2, dtype=torch.float32, device=device)
    problem = layout.problem(device, runs, scale, query.dtype, d, kvb, tabs)
    check_tables(layout, problem, host, device, tabs)
    keep = [keep_runs]
    ds = _ds_route(layout, query, lib)
    if ds is not None:
        _, kv_heads = ds
        group = layout.hq // layout.hkv
        try:
            work = torch.empty(kv_heads * group * tabs["head"] + 512, dtype=query.dtype, device=device)
        except torch.cuda.OutOfMemoryError:
            ds = None
    with operator_range("hip_attention_backward", rows=layout.q_rows, segments=len(layout.seg_q),
                        ds_route=ds is not None):
        if ds is None:
            _lib.check(
                lib.ts_attn_bwd(ctypes.byref(problem), _rows(query), _rows(out), _rows(dout),
                                lse.data_ptr(), lse.shape[1], rowstats.data_ptr(), _rows(dq),
                                _lib.stream_of(query)),
                lambda: f"ts_attn_bwd(rows={layout.q_rows}, hq={layout.hq}, hkv={layout.hkv})",
            )
        else:
            rows = [_rows(t) for t in (query, out, dout, dq)]
            # the dQ pass's 64-row list where it applies (head dim 128, groups of 4)
            dq_list, n_dq, n_dq_long = None, 0, 0
            if d == HEAD_DIM and tabs["dq_work"] is not None:
                dq_list, n_dq, n_dq_long = tabs["dq_work"], tabs["n_dq_work"], tabs["n_dq_long"]
            # the whole problem's parts for every group of KV heads: the same sums either way
            parts = lib.ts_attn_dq_parts(ctypes.byref(problem), n_dq, desc["max_keys"])
            for hk0 in range(0, layout.hkv, kv_heads):
                n, h0 = min(kv_heads, layout.hkv - hk0), hk0 * group
                sub = problem
                if n != layout.hkv:  # KV heads hk0 .. hk0 + n - 1 and their query heads
                    sub_runs, sub_host = _head_runs(host, hk0, device)
                    keep.append((sub_runs, sub_host))
                    sub = AttnProblem.from_buffer_copy(problem)
                    sub.hq, sub.hkv, sub.runs = n * group, n, sub_runs.data_ptr()
                    check_tables(layout, sub, sub_host, device, tabs)
                q_r, o_r, do_r, dq_r = (_head_rows(r, h0) for r in rows)
                sums = None
                if parts > 1:
                    sums = _parts_workspace(lib.ts_attn_dq_parts_workspace(ctypes.byref(sub), n_dq, parts), device)
                    parts = parts if sums is not None else 1
                _lib.check(
                    lib.ts_attn_bwd_ds_split(ctypes.byref(sub), q_r, o_r, do_r, lse.data_ptr() + h0 * lse.shape[1] * 4,
                                       lse.shape[1], rowstats.data_ptr() + h0 * lse.shape[1] * 8, dq_r,
                                       tabs["span"], tabs["visit"], tabs["head"], work.data_ptr(),
                                       work.numel() * 2, dq_list, n_dq, n_dq_long, parts, _lib.ptr(sums),
                                       0 if sums is None else sums.numel(), _lib.stream_of(query)),
                    lambda: f"ts_attn_bwd_ds(rows={layout.q_rows}, hq={layout.hq}, hkv={layout.hkv}, heads from {h0})",
                )
            del work
    count_attention_path(HIP_BACKWARD_PATH)
    return dq, dkeys, dvalues, keep


class _Attention(torch.autograd.Function):
    """out, lse = attention over `layout`; grads to query and every key source."""

    @staticmethod
    def forward(ctx, query, layout, scale, n_sources, *kv):
        out, lse, ctx.keep = _attention_forward(query, layout, scale, kv[:n_sources], kv[n_sources:])
        ctx.layout, ctx.scale, ctx.n_sources = layout, scale, n_sources
        ctx.save_for_backward(query, out, lse, *kv)
        ctx.mark_non_differentiable(lse)
        ctx.set_materialize_grads(False)  # no zero-filled gradient for lse
        return out, lse

    @staticmethod
    @torch.autograd.function.once_differentiable
    def backward(ctx, dout, _dlse):
        query, out, lse, *kv = ctx.saved_tensors
        if dout is None:
            dout = torch.zeros_like(out)
        n = ctx.n_sources
        dq, dkeys, dvalues, ctx.keep_bwd = _attention_backward(query, out, lse, dout, ctx.layout, ctx.scale, kv[:n],
                                                               kv[n:])
        return (dq, None, None, None, *dkeys, *dvalues)


def kernel_head_dim(head_dim: int) -> int | None:
    """The kernel head dim that runs `head_dim`: itself when the kernels are
    built for it, else the next larger one (for 1 <= head_dim <= 256), None
    above 256.  Zero columns appended to Q and K change no score and zero
    columns of V only add output columns, so the padded call's output and
    gradients restricted to the first `head_dim` columns are the unpadded
    ones; the caller's scale is used as given."""
    if head_dim < 1:
        return None
    for d in HEAD_DIMS:
        if head_dim <= d:
            return d
    return None


def attention(query: torch.Tensor, layout: AttnLayout, keys: Sequence[torch.Tensor],
              values: Sequence[torch.Tensor], scale: float) -> tuple[torch.Tensor, torch.Tensor]:
    """Core op: query ``[R, Hq, D]`` bf16 or fp16 -> (out ``[R, Hq, D]``, lse ``[Hq, R]`` fp32).

    A head dim the kernels are not built for (any other D up to 256) runs at
    :func:`kernel_head_dim` over zero-padded copies of Q, K and V; autograd
    takes the gradients back through the padding."""
    d = query.shape[-1] if query.dim() == 3 else -1
    dk = kernel_head_dim(d)
    if dk is not None and dk != d:
        def pad(t):
            return torch.nn.functional.pad(t, (0, dk - t.shape[-1]))
        out, lse = _Attention.apply(pad(query), layout, float(scale), len(keys), *(pad(k) for k in keys),
                                    *(pad(v) for v in values))
        return out[..., :d], lse
    return _Attention.apply(query, layout, float(scale), len(keys), *keys, *values)


def _pad_heads(t: torch.Tensor, head_dim: int) -> torch.Tensor:
    return torch.nn.functional.pad(t, (0, head_dim - t.shape[-1])) if t.shape[-1] != head_dim else t


def _save_attention(ctx, query: torch.Tensor, layout: AttnLayout, scale: float, keys, values) -> torch.Tensor:
    """The forward of an autograd function that differentiates the core op
    itself (no graph inside it): out ``[R, Hq, D]``, with everything
    :func:`_saved_gradients` needs saved on ``ctx``.  Head dims as in
    :func:`attention`."""
    d = query.shape[-1]
    dk = kernel_head_dim(d) or d
    if dk != d:  # else keys and values of another head dim are refused below
        query, keys, values = _pad_heads(query, dk), [_pad_heads(k, dk) for k in keys], [_pad_heads(v, dk) for v in values]
    out, lse, ctx.keep = _attention_forward(query, layout, float(scale), keys, values)
    ctx.layout, ctx.scale = layout, float(scale)
    ctx.save_for_backward(query, out, lse, *keys, *values)
    return out[..., :d] if dk != d else out


def _saved_gradients(ctx, dout: torch.Tensor):
    """(dq, dkeys, dvalues) of a call saved by :func:`_save_attention`, for the
    gradient ``[R, Hq, D]`` of its output."""
    query, out, lse, *kv = ctx.saved_tensors
    d, n = dout.shape[-1], len(kv) // 2
    dq, dkeys, dvalues, ctx.keep_bwd = _attention_backward(query, out, lse, _pad_heads(dout, query.shape[-1]),
                                                           ctx.layout, ctx.scale, kv[:n], kv[n:])
    if query.shape[-1] != d:
        # dense gradients that do not keep the padded ones
        dq, *rest = (g[..., :d].clone() for g in (dq, *dkeys, *dvalues))
        dkeys, dvalues = rest[:n], rest[n:]
    return dq, dkeys, dvalues


# ---------------------------------------------------------------------------
# layouts for the reference's call shapes
# ---------------------------------------------------------------------------
def chain_layout(query_len: int, chunk_lengths: Sequence[int], hq: int, hkv: int) -> AttnLayout:
    """One segment of `query_len` rows over the concatenation of chunks."""
    runs, spans, pos = [], [], 0
    for i, n in enumerate(chunk_lengths):
        if n > 0:
            spans.append((len(runs), pos))
            runs.append(Run(i, 0, n))
            pos += n
    return AttnLayout(
        q_rows=query_len, hq=hq, hkv=hkv, source_rows=tuple(chunk_lengths), runs=tuple(runs),
        seg_q=((0, query_len),), seg_spans=(tuple(spans),),
    )


def _query_rows(query: torch.Tensor) -> torch.Tensor:
    """``[1, Hq, T, D]`` (any strides) -> ``[T, Hq, D]`` view."""
    if query.dim() != 4 or query.shape[0] != 1:
        raise ValueError(f"query must be [1, Hq, T, D], got {tuple(query.shape)}")
    # squeeze, not select: the gradient of a select is a zero-filled copy
    return query.squeeze(0).transpose(0, 1)


def _as_rows(t: torch.Tensor) -> torch.Tensor:
    """A [rows, heads, D] view usable by the kernels (copy only if it must)."""
    s = t.stride()
    if s[2] == 1 and not (s[0] | s[1]) & 7 and not t.data_ptr() & 15:
        return t
    return t.contiguous()


def causal_attention(query: torch.Tensor, ks: Sequence[torch.Tensor], vs: Sequence[torch.Tensor],
                     scale: float) -> torch.Tensor:
    """Backend callable ``(query [1,Hq,T,D], ks, vs, scale) -> [1,Hq,T,D]``.

    ``ks``/``vs`` are chunk lists ``[S_c, Hkv, D]`` in chronological order;
    query row i sees keys ``0 .. S - T + i`` of their concatenation, which is
    never materialised (engine/streaming.py:1080-1162).
    """
    q, layout, keys, values = _chain_call(query, ks, vs)
    out, _ = attention(q, layout, keys, values, scale)
    return out.transpose(0, 1).unsqueeze(0)


def _chain_call(query, ks, vs):
    """(query rows, layout, keys, values) of a chunk-list call, one run per chunk."""
    q = _as_rows(_query_rows(query))
    keys = [_as_rows(k) for k in ks]
    values = [_as_rows(v) for v in vs]
    return q, chain_layout(q.shape[0], [k.shape[0] for k in keys], q.shape[1], keys[0].shape[1]), keys, values


class ChunkedCausalAttention(torch.autograd.Function):
    """``apply(query, scale, n_chunks, keep_state, backend, *ks, *vs)``.

    Argument order and meaning of ``_ChunkedCausalSDPA`` (engine/streaming.py:
    1314-1423): bottom-right-causal attention of ``query [1, Hq, T, D]`` over
    the chunk lists as one op that keeps only references to the per-chunk K/V
    (never a concatenated copy) and returns one dK/dV per chunk in input order.

    * ``backend`` ``"auto"`` or ``"cudnn"`` (the reference's built-in names):
      the HIP kernels.  The op keeps the query, its output and log-sum-exp --
      what the reference's saved-state mode keeps -- and its backward runs
      the HIP backward on them, whatever ``keep_state`` says (the reference's
      other mode re-runs the forward to reach the same numbers; the HIP
      forward is deterministic, so keeping them is equivalent).
    * a callable ``backend(query, ks, vs, scale)``: called as the reference
      calls it (:1094-1095), and differentiated by re-running it under
      autograd in the backward (:1384-1399).
    * any other name raises ``ValueError`` (:1096-1097).
    """

    @staticmethod
    def forward(ctx, query, scale, n_chunks, keep_state, backend, *chunks):
        ks, vs = list(chunks[:n_chunks]), list(chunks[n_chunks:])
        ctx.n_chunks, ctx.scale, ctx.backend = n_chunks, scale, backend
        if callable(backend):
            ctx.save_for_backward(query, *chunks)
            return backend(query, ks, vs, scale)
        if backend not in ("auto", "cudnn"):
            raise ValueError(f"unknown source attention backend: {backend!r}")
        q, layout, keys, values = _chain_call(query, ks, vs)
        out = _save_attention(ctx, q, layout, scale, keys, values)
        return out.transpose(0, 1).unsqueeze(0).detach()

    @staticmethod
    @torch.autograd.function.once_differentiable
    def backward(ctx, grad_out):
        need = ctx.needs_input_grad
        n = ctx.n_chunks
        if callable(ctx.backend):
            query, *chunks = ctx.saved_tensors
            q = query.detach().requires_grad_(True)
            leaves = [c.detach().requires_grad_(True) for c in chunks]
            with torch.enable_grad():
                out = ctx.backend(q, leaves[:n], leaves[n:], ctx.scale)
            grads = torch.autograd.grad(out, [q, *leaves], grad_out, allow_unused=True)
            dq, rest = grads[0], list(grads[1:])
        else:
            dq, dkeys, dvalues = _saved_gradients(ctx, grad_out[0].transpose(0, 1))
            dq = dq.transpose(0, 1).unsqueeze(0)
            rest = [*dkeys, *dvalues]
        return (
            dq if need[0] else None, None, None, None, None,
            *(g if need[5 + i] else None for i, g in enumerate(rest)),
        )


@dataclass(eq=False)
class PackLayout:
    """Where each segment of a plain turn pack sits (engine/streaming.py:1613-1650).

    ``lengths``: query rows per segment; ``prefixes``: ancestor tokens per
    segment; ``counts``: ancestor chunks per segment.  ``cu_lengths`` and
    ``cu_prefixes`` are the int32 cumulative sums ``[0, *accumulate(...)]``.
    The op's ancestor inputs are grouped by segment, LAST segment first.
    """

    lengths: list[int]
    prefixes: list[int]
    counts: list[int]
    cu_lengths: torch.Tensor
    cu_prefixes: torch.Tensor
    counted: bool = True

    def inputs(self, ancestors):
        ks = [c for ks, _vs in reversed(ancestors) for c in ks]
        vs = [c for _ks, vs in reversed(ancestors) for c in vs]
        return ks + vs

    def by_segment(self, chunks):
        grouped, offset = [], 0
        for count in reversed(self.counts):
            grouped.append(list(chunks[offset : offset + count]))
            offset += count
        return grouped[::-1]


def pack_layout(lengths: Sequence[int], ancestors, device=None) -> PackLayout:
    """Build a PackLayout from per-segment lengths and ancestor chunk lists."""
    from itertools import accumulate

    prefixes = [sum(c.shape[0] for c in ks) for ks, _vs in ancestors]
    counts = [len(ks) for ks, _vs in ancestors]
    cu_l = torch.tensor([0, *accumulate(lengths)], dtype=torch.int32)
    cu_p = torch.tensor([0, *accumulate(prefixes)], dtype=torch.int32)
    if device is not None and torch.device(device).type == "cuda":
        cu_l = cu_l.pin_memory().to(device, non_blocking=True)
        cu_p = cu_p.pin_memory().to(device, non_blocking=True)
    return PackLayout(list(lengths), prefixes, counts, cu_l, cu_p)


class PackedAttention(torch.autograd.Function):
    """``apply(query, key, value, scale, layout, *ancestors)``, as _PackedFlashSplit.

    ``query [1, Hq, sum(T), D]``, the pack's own ``key``/``value`` ``[sum(T),
    Hkv, D]``, then the ancestor chunks in ``PackLayout.inputs`` order.  Each
    segment attends to its ancestors (fully) then its own rows (causally);
    one forward and one backward launch serve the whole pack.  A chunk object
    passed for several segments (the shared prompt) is one key run visited
    by each of them, so its gradient is summed inside the kernel.
    """

    @staticmethod
    def forward(ctx, query, key, value, scale, layout, *ancestors):
        total = sum(layout.counts)
        a_keys = layout.by_segment(ancestors[:total])
        a_vals = layout.by_segment(ancestors[total:])
        q = _as_rows(_query_rows(query))
        own_k, own_v = _as_rows(key), _as_rows(value)
        srcs_k, srcs_v, src_index = [own_k], [own_v], {}
        runs: list[Run] = []
        seg_q, seg_spans = [], []
        row0 = 0
        # own-K/V runs, one per segment (source 0)
        own_runs = []
        for length in layout.lengths:
            own_runs.append(len(runs))
            runs.append(Run(0, row0, length))
            row0 += length
        chunk_run = {}
        for s, (length, ks, vs) in enumerate(zip(layout.lengths, a_keys, a_vals)):
            spans, pos = [], 0
            for kc, vc in zip(ks, vs):
                if kc.shape[0] == 0:
                    continue
                ident = (id(kc), id(vc))
                if ident not in chunk_run:
                    if ident not in src_index:
                        src_index[ident] = len(srcs_k)
                        srcs_k.append(_as_rows(kc))
                        srcs_v.append(_as_rows(vc))
                    chunk_run[ident] = len(runs)
                    runs.append(Run(src_index[ident], 0, kc.shape[0]))
                spans.append((chunk_run[ident], pos))
                pos += kc.shape[0]
            if length > 0:
                spans.append((own_runs[s], pos))
            seg_q.append((sum(layout.lengths[:s]), length))
            seg_spans.append(tuple(spans))
        att_layout = AttnLayout(
            q_rows=q.shape[0], hq=q.shape[1], hkv=own_k.shape[1],
            source_rows=tuple(t.shape[0] for t in srcs_k), runs=tuple(runs),
            seg_q=tuple(seg_q), seg_spans=tuple(seg_spans),
        )
        out = _save_attention(ctx, q, att_layout, scale, srcs_k, srcs_v)
        # per ancestor input, in input order: its source, or None for an empty
        # chunk (zeros) or a repeated one (whose gradient the first carries)
        order, seen = [], set()
        for ks, vs in zip(reversed(a_keys), reversed(a_vals)):
            for kc, vc in zip(ks, vs):
                ident = (id(kc), id(vc))
                source = src_index.get(ident) if kc.shape[0] and ident not in seen else None
                order.append((source, kc.shape[0] == 0, kc.shape, vc.shape))
                seen.add(ident)
        ctx.order = order
        return out.detach().transpose(0, 1).unsqueeze(0)

    @staticmethod
    @torch.autograd.function.once_differentiable
    def backward(ctx, grad_out):
        dq, dks, dvs = _saved_gradients(ctx, grad_out[0].transpose(0, 1))
        # ancestor grads in input order; a chunk object appearing several
        # times receives its summed gradient once (autograd adds per input)
        anc_k, anc_v = [], []
        for source, empty, k_shape, v_shape in ctx.order:
            if source is not None:
                anc_k.append(dks[source])
                anc_v.append(dvs[source])
            else:
                anc_k.append(torch.zeros(k_shape, dtype=dq.dtype, device=dq.device) if empty else None)
                anc_v.append(torch.zeros(v_shape, dtype=dq.dtype, device=dq.device) if empty else None)
        return (dq.transpose(0, 1).unsqueeze(0) if ctx.needs_input_grad[0] else None, dks[0], dvs[0], None, None,
                *anc_k, *anc_v)


def _ragged_layout(lengths: Sequence[int], key_rows: Sequence[int], hq: int, hkv: int) -> AttnLayout:
    """Segment i: ``lengths[i]`` packed query rows over key source i alone."""
    runs = tuple(Run(i, 0, n) for i, n in enumerate(key_rows))
    seg_q, row0 = [], 0
    for n in lengths:
        seg_q.append((row0, n))
        row0 += n
    return AttnLayout(
        q_rows=row0, hq=hq, hkv=hkv, source_rows=tuple(key_rows), runs=runs,
        seg_q=tuple(seg_q), seg_spans=tuple(((i, 0),) for i in range(len(key_rows))),
    )


def ragged_causal_attention(queries, keys, values, scale):
    """``_ragged_causal_sdpa`` (engine/streaming.py:1165-1226): per segment
    ``[1,Hq,T_i,D]`` over its own ``[S_i,Hkv,D]``, bottom-right causal, all
    segments in one launch.  Differentiable (one backward launch)."""
    if not queries:
        return []
    q_rows = [_as_rows(_query_rows(q)) for q in queries]
    lengths = [q.shape[0] for q in q_rows]
    packed = torch.cat(q_rows, 0)
    srcs_k = [_as_rows(k) for k in keys]
    srcs_v = [_as_rows(v) for v in values]
    layout = _ragged_layout(lengths, [k.shape[0] for k in srcs_k], packed.shape[1], srcs_k[0].shape[1])
    out, _ = attention(packed, layout, srcs_k, srcs_v, scale)
    return [piece.transpose(0, 1).unsqueeze(0) for piece in out.split(lengths, 0)]


class RaggedAttention(torch.autograd.Function):
    """``apply(scale, n_segments, *queries, *keys, *values)`` -> one output per
    segment, as ``_RaggedAttentionIndependentVJP`` (engine/streaming.py:
    1253-1297).  The reference runs the cohort through one varlen flash call
    and recomputes each segment with ``_causal_sdpa`` in its backward; here
    the forward is one HIP launch for the cohort and the backward one HIP
    backward launch over the saved output and log-sum-exp, which gives every
    segment its own independent VJP (segments share no keys)."""

    @staticmethod
    def forward(ctx, scale, n_segments, *tensors):
        queries = list(tensors[:n_segments])
        keys = list(tensors[n_segments : 2 * n_segments])
        values = list(tensors[2 * n_segments :])
        with torch.enable_grad():
            qs = [q.detach().requires_grad_(q.requires_grad) for q in queries]
            kk = [k.detach().requires_grad_(k.requires_grad) for k in keys]
            vv = [v.detach().requires_grad_(v.requires_grad) for v in values]
            outs = ragged_causal_attention(qs, kk, vv, scale)
        ctx.graph = (qs + kk + vv, outs)
        return tuple(o.detach() for o in outs)

    @staticmethod
    @torch.autograd.function.once_differentiable
    def backward(ctx, *grad_outputs):
        leaves, outs = ctx.graph
        inputs = [t for t in leaves if t.requires_grad]
        grads = torch.autograd.grad(outs, inputs, grad_outputs, allow_unused=True) if inputs else []
        it = iter(grads)
        return (None, None, *(next(it) if t.requires_grad else None for t in leaves))


# ---------------------------------------------------------------------------
# retained chunks
# ---------------------------------------------------------------------------
def retained_chunk_layout(q_rows: int, chunk_rows: Sequence[int], chunks: Sequence[tuple[int, int, Sequence[int]]],
                          hq: int, hkv: int) -> AttnLayout:
    """Query chunks over graph-retained per-chunk K/V, all in one launch.

    ``chunk_rows[i]`` is the row count of retained chunk ``i`` (one K and one
    V tensor each); ``chunks`` lists every query chunk as ``(q_row0, q_len,
    path)`` where ``path`` names, in key order, the retained chunks the query
    chunk reads -- the prompt's chunks, the earlier chunks of its trajectory
    and its own chunk last.  Each query chunk is the bottom-right-causal call
    ``_ChunkedCausalSDPA`` makes per chunk (engine/streaming.py:1314-1354);
    the retained tensors are read in place, never concatenated.
    """
    runs = tuple(Run(i, 0, n) for i, n in enumerate(chunk_rows))
    seg_q, seg_spans = [], []
    for row0, length, path in chunks:
        spans, pos = [], 0
        for c in path:
            if not 0 <= c < len(runs):
                raise ValueError(f"query chunk at row {row0} names retained chunk {c} of {len(runs)}")
            spans.append((c, pos))
            pos += runs[c].length
        seg_q.append((row0, length))
        seg_spans.append(tuple(spans))
    return AttnLayout(q_rows=q_rows, hq=hq, hkv=hkv, source_rows=tuple(chunk_rows), runs=runs,
                      seg_q=tuple(seg_q), seg_spans=tuple(seg_spans))


def retained_chunk_attention(query: torch.Tensor, ks: Sequence[torch.Tensor], vs: Sequence[torch.Tensor],
                             layout: AttnLayout, scale: float) -> torch.Tensor:
    """``query`` ``[R, Hq, D]`` over retained chunks ``ks``/``vs`` (each
    ``[S_c, Hkv, D]``) as described by :func:`retained_chunk_layout`;
    differentiable wrt the query and every retained chunk."""
    out, _ = attention(_as_rows(query), layout, [_as_rows(k) for k in ks], [_as_rows(v) for v in vs], scale)
    return out


# ---------------------------------------------------------------------------
# forest
# ---------------------------------------------------------------------------
def forest_layout(plan, hq: int, hkv: int) -> AttnLayout:
    """Segments = non-empty nodes, runs = node ranges of the one K/V tensor.

    ``plan`` is an ExecutionPlan (engine/plan.py:41-73) or anything with
    ``node_start``, ``node_end`` (per node) and ``key_ranges`` (per node:
    ancestor spans then the node's own span, engine/plan.py:248-256).
    """
    cached = getattr(plan, "_thundersync_hip_layouts", None)
    if cached is not None and (hq, hkv) in cached:
        return cached[(hq, hkv)]
    starts = [int(x) for x in plan.node_start.tolist()]
    ends = [int(x) for x in plan.node_end.tolist()]
    p = int(plan.n_physical) if hasattr(plan, "n_physical") else max(ends, default=0)
    run_of_start = {}
    runs = []
    for n, (s, e) in enumerate(zip(starts, ends)):
        if e > s:
            run_of_start[(s, e)] = len(runs)
            runs.append(Run(0, s, e - s))
    order = sorted((n for n in range(len(starts)) if ends[n] > starts[n]), key=lambda n: starts[n])
    seg_q, seg_spans = [], []
    for n in order:
        spans, pos = [], 0
        for s, e in plan.key_ranges[n]:
            if e <= s:
                continue
            if (s, e) not in run_of_start:
                raise ValueError(f"key range ({s}, {e}) of node {n} is not a node range")
            spans.append((run_of_start[(s, e)], pos))
            pos += e - s
        seg_q.append((starts[n], ends[n] - starts[n]))
        seg_spans.append(tuple(spans))
    layout = AttnLayout(
        q_rows=p, hq=hq, hkv=hkv, source_rows=(p,), runs=tuple(runs),
        seg_q=tuple(seg_q), seg_spans=tuple(seg_spans),
    )
    try:
        if cached is None:
            cached = {}
            object.__setattr__(plan, "_thundersync_hip_layouts", cached)
        cached[(hq, hkv)] = layout
    except (AttributeError, TypeError):
        pass
    return layout


def forest_attention(q: torch.Tensor, k: torch.Tensor, v: torch.Tensor, plan, *, scale: float | None = None):
    """Attention over a segment forest on the physical stream (engine/attention.py:186-231).

    ``q`` ``[P, Hq, D]``, ``k``/``v`` ``[P, Hkv, D]``; returns ``[P, Hq, D]``.
    Every node attends to its ancestors in full and to itself causally, in
    one launch per direction; no mask and no ancestor concatenation.
    """
    scale = scale if scale is not None else 1.0 / math.sqrt(q.shape[-1])
    if q.shape[1] % k.shape[1]:
        raise ValueError(f"query heads {q.shape[1]} are not divisible by KV heads {k.shape[1]}")
    layout = forest_layout(plan, q.shape[1], k.shape[1])
    out, _ = attention(_as_rows(q), layout, [_as_rows(k)], [_as_rows(v)], scale)
    return out


# ---------------------------------------------------------------------------
# transformers AttentionInterface adapters
# ---------------------------------------------------------------------------
HIP_ATTENTION_NAME = "thundersync_hip"
HIP_FOREST_ATTENTION_NAME = "thundersync_hip_forest"
_PLANS: dict[torch.device, object] = {}


def hip_attention_forward(module, query, key, value, attention_mask, scaling=None, dropout=0.0, **kwargs):
    """Causal attention over one sequence, heads last on the way out.

    The signature and contract of ``fa4_attention_forward``
    (accel/fa4_attention.py:22-53): ``[B, H, T, D]`` in, ``[B, T, H, D]``
    out, grouped K/V heads carried natively, dropout refused.
    """
    if dropout:
        raise ValueError("attention dropout is not supported on this path")
    scale = scaling if scaling is not None else query.shape[-1] ** -0.5
    if query.shape[0] == 1:
        # views whose gradients are views too (an indexed batch row's gradient
        # would be a zero-filled copy of the whole batch)
        o = causal_attention(query, [key.squeeze(0).transpose(0, 1)], [value.squeeze(0).transpose(0, 1)], scale)
        return o.transpose(1, 2), None
    outs = []
    for qb, kb, vb in zip(query.unbind(0), key.unbind(0), value.unbind(0)):
        o = causal_attention(qb.unsqueeze(0), [kb.transpose(0, 1)], [vb.transpose(0, 1)], scale)
        outs.append(o.transpose(1, 2))
    return torch.cat(outs, 0), None


def forest_attention_forward(module, query, key, value, attention_mask, dropout=0.0, scaling=None, **kwargs):
    """HF adapter of engine/step.py:60-99 over the plan bound by :func:`forest_context`."""
    plan = _PLANS.get(query.device)
    if plan is None:
        raise RuntimeError("forest attention was invoked outside `forest_context`")
    if query.shape[0] != 1:
        raise ValueError(f"the forest is already the batch; expected batch dim 1, got {query.shape[0]}")
    out = forest_attention(query.squeeze(0).transpose(0, 1), key.squeeze(0).transpose(0, 1),
                           value.squeeze(0).transpose(0, 1), plan, scale=scaling)
    return out.unsqueeze(0), None


class forest_context:
    """Bind a plan for the duration of a forward (and backward), per device."""

    def __init__(self, plan, device=None):
        self.plan = plan
        self.device = torch.device(device) if device is not None else plan.token_ids.device

    def __enter__(self):
        self.previous = _PLANS.get(self.device)
        _PLANS[self.device] = self.plan
        return self.plan

    def __exit__(self, *exc):
        if self.previous is None:
            _PLANS.pop(self.device, None)
        else:
            _PLANS[self.device] = self.previous
        return False


def register_attention() -> bool:
    """Register both adapters with transformers' AttentionInterface."""
    try:
        from transformers.modeling_utils import AttentionInterface
    except Exception:
        return False
    AttentionInterface.register(HIP_ATTENTION_NAME, hip_attention_forward)
    AttentionInterface.register(HIP_FOREST_ATTENTION_NAME, forest_attention_forward)
    return True
