"""Batch of estimator instances, packed into one float64 arena in HBM.

A ``Batch`` collects already validated and rescaled columns (NumPy float64)
and estimator instances that reference them.  Columns passed as the same
NumPy object are stored once, so instances that share a column (the x role
of one variable across ``pairwise_mi`` pairs, say) also share its device sort.
``Batch.run`` uploads the arena through PyTorch-ROCm, runs every instance in
one ``enm_run_batch`` call and returns one float64 value per instance.
"""

from __future__ import annotations

import ctypes
import functools
import itertools
import threading
from typing import Dict, List, Optional, Sequence, Tuple

import numpy as np

from . import _native as nat


class Batch:
    def __init__(self) -> None:
        self._cols: List[np.ndarray] = []
        self._orig: List[np.ndarray] = []
        self._col_index: Dict[int, int] = {}
        self._inst: List[tuple] = []
        self._seg: List[int] = []

    def __len__(self) -> int:
        return len(self._inst)

    def _col(self, a: np.ndarray) -> int:
        # The originals are kept alive, so an id() cannot be reused meanwhile.
        key = id(a)
        idx = self._col_index.get(key)
        if idx is None:
            c = np.asarray(a, dtype=np.float64)
            if c.ndim != 1:
                raise ValueError("columns must be one-dimensional")
            idx = len(self._cols)
            self._cols.append(c)
            self._orig.append(a)
            self._col_index[key] = idx
        return idx

    def add(self, kind: int, k: int, x: Sequence[np.ndarray], y: Sequence[np.ndarray] = (),
            z: Sequence[np.ndarray] = (), class_sizes: Optional[Sequence[int]] = None) -> int:
        """Add one instance; returns its index.  For ROSS/CROSS the points must
        be grouped by class, in class order, with the given class sizes."""
        cols = [self._col(c) for c in list(x) + list(y) + list(z)]
        if len(cols) > nat.MAX_COLS:
            raise ValueError(f"at most {nat.MAX_COLS} dimensions per instance")
        n = len(self._cols[cols[0]])
        for c in cols:
            if len(self._cols[c]) != n:
                raise ValueError("all columns of an instance must have the same length")
        seg_index = len(self._seg)
        if class_sizes is None:
            n_segs = 1
        else:
            n_segs = len(class_sizes)
            self._seg.extend(int(s) for s in class_sizes)
        self._inst.append((kind, int(k), n, len(x), len(y), len(z), n_segs, seg_index, cols))
        return len(self._inst) - 1

    def pack(self):
        """The ctypes instance / class-size tables; columns lie one after the other."""
        offsets = np.cumsum([0] + [len(c) for c in self._cols])
        inst_arr = _instance_table(self._inst, offsets)
        seg_arr = (ctypes.c_int64 * max(1, len(self._seg)))(*self._seg)
        return inst_arr, seg_arr

    def arena(self, device, stream):
        """The columns in HBM, sent up on `stream`; returns (arena, pinned host copy)."""
        return upload_columns(self._cols, device, stream)

    def point_offsets(self) -> np.ndarray:
        n = np.array([t[2] for t in self._inst], dtype=np.int64)
        return np.concatenate([[0], np.cumsum(n)])

    def device(self, flags: int = 0, export: bool = False):
        """Upload the arena; return a DeviceBatch ready to launch."""
        return DeviceBatch(self, flags, export)

    def run(self, flags: int = 0, export: bool = False):
        """Run every instance.  Returns values, or (values, eps, counts) with
        per-instance lists of radii (n,) and counts (3, n) when export=True."""
        with on(_stream()):
            db = self.device(flags, export)
            db.launch()
            return db.results()


def _instance_table(inst: List[tuple], col_offsets: Optional[np.ndarray]):
    """The ctypes enm_instance table of (kind, k, n, dx, dy, dz, n_segs,
    seg_index, columns) tuples; a column is an arena offset, or an index
    into col_offsets."""
    n_inst = len(inst)
    inst_arr = (nat.EnmInstance * n_inst)()
    if n_inst == 0:
        return inst_arr
    tab = nat.struct_array(inst_arr)
    head = np.array([t[:8] for t in inst], dtype=np.int64).reshape(n_inst, 8)
    for f, name in enumerate(("kind", "k", "n", "dx", "dy", "dz", "n_segs", "seg_index")):
        tab[name] = head[:, f]
    width = max(len(t[8]) for t in inst)
    cols = np.zeros((n_inst, width), dtype=np.int64)
    for i, t in enumerate(inst):
        cols[i, :len(t[8])] = t[8]
    if col_offsets is not None:
        cols = np.where(np.arange(width) < np.array([len(t[8]) for t in inst])[:, None], col_offsets[cols], 0)
    tab["col"][:, :width] = cols
    return inst_arr


class DeviceBatch:
    """A packed batch resident in HBM, launchable many times (bench, graphs)."""

    def __init__(self, batch: Batch, flags: int, export: bool, hints: bool = True):
        import torch
        self.batch = batch
        # Sort hints of a device-prepared arena (enm_run_batch_hinted).
        self.hint = getattr(batch, "device_hint", None) if hints else None
        self.ctx = nat.context()
        self.flags = flags
        self.inst_arr, self.seg_arr = batch.pack()
        self.n_inst = len(batch)
        dev = torch.device("cuda", self.ctx.device)
        self.stream = _stream()
        with on(self.stream):
            self.arena, self._pinned = batch.arena(dev, self.stream)
            self.out = torch.empty(self.n_inst, dtype=torch.float64, device=dev)
            self.offs = batch.point_offsets()
            total = int(self.offs[-1])
            self.eps = torch.empty(total, dtype=torch.float64, device=dev) if export else None
            self.counts = torch.empty(3 * total, dtype=torch.int32, device=dev) if export else None

    def launch(self) -> None:
        """Enqueue one run on the batch's stream (returns immediately)."""
        with self.ctx.lock:
            self.ctx.run(self.inst_arr, self.n_inst, self.seg_arr, self.arena.data_ptr(),
                         self.out.data_ptr(), self.eps.data_ptr() if self.eps is not None else 0,
                         self.counts.data_ptr() if self.counts is not None else 0,
                         self.flags, self.stream.cuda_stream,
                         self.hint.data_ptr() if self.hint is not None else 0)

    def stats(self) -> dict:
        with self.ctx.lock:
            return self.ctx.stats()

    def autotune(self) -> Tuple[int, int]:
        """Time the library's tile shapes on this batch and keep the fastest
        (in the context, for every later batch); returns (strip, waves/CU)."""
        with self.ctx.lock:
            self.ctx.autotune(self.inst_arr, self.n_inst, self.seg_arr, self.arena.data_ptr(),
                              self.out.data_ptr(), self.flags, self.stream.cuda_stream)
            self.stream.synchronize()
            return self.ctx.get_tuning()

    def results(self):
        import torch
        with on(self.stream):
            host = torch.empty(self.n_inst, dtype=torch.float64, pin_memory=True).copy_(self.out, non_blocking=True)
        self.stream.synchronize()
        values = host.numpy().copy()
        if self.eps is None:
            return values
        eps_all = self.eps.cpu().numpy()
        cnt_all = self.counts.cpu().numpy()
        eps, cnts = [], []
        for i in range(self.n_inst):
            a, b = int(self.offs[i]), int(self.offs[i + 1])
            n = b - a
            eps.append(eps_all[a:b].copy())
            cnts.append(cnt_all[3 * a:3 * b].reshape(3, n).copy())
        return values, eps, cnts


class ArenaBatch:
    """A batch whose float64 arena was written on the device (the columns
    of device-prepared tasks, enm_prep_write), with the sort hints of its
    columns when they were made (enm_prep_hints); instances name their
    columns by arena offset.  Same interface as Batch."""

    def __init__(self, device_arena, device_hint=None) -> None:
        self.device_arena = device_arena
        self.device_hint = device_hint
        self._runs: List[tuple] = []   # (kind, k, n per instance, dx, dy, dz, offsets per instance)
        self._classes = None           # class sizes per instance (Ross kinds): n_segs, seg_index, all sizes

    def __len__(self) -> int:
        return sum(len(r[2]) for r in self._runs)

    def add(self, kind: int, k: int, n: int, offsets: Sequence[int], dx: int, dy: int, dz: int) -> int:
        self.add_many(kind, k, [n], [offsets], dx, dy, dz)
        return len(self) - 1

    def add_many(self, kind: int, k: int, n, offsets, dx: int, dy: int, dz: int) -> None:
        """Instances of one kind: their points n (per instance) and column
        offsets (per instance and column)."""
        self._runs.append((kind, int(k), np.asarray(n, dtype=np.int64), dx, dy, dz,
                           np.asarray(offsets, dtype=np.int64)))

    def set_classes(self, sizes: np.ndarray) -> None:
        """Rows of every class (instances by classes, 0: none) of the Ross
        instances that are the whole batch."""
        n_segs = (sizes > 0).sum(axis=1)
        self._classes = (n_segs, np.cumsum(n_segs) - n_segs, sizes[sizes > 0])

    @property
    def _inst(self) -> List[tuple]:
        n_segs, seg_index = self._classes[:2] if self._classes is not None else (itertools.repeat(1), itertools.repeat(0))
        head = ((kind, k, int(n), dx, dy, dz, [int(o) for o in offs])
                for kind, k, ns, dx, dy, dz, cols in self._runs for n, offs in zip(ns, cols))
        return [(*h[:6], int(m), int(first), h[6]) for h, m, first in zip(head, n_segs, seg_index)]

    def pack(self):
        inst_arr = (nat.EnmInstance * len(self))()
        tab = nat.struct_array(inst_arr)
        at = 0
        for kind, k, n, dx, dy, dz, cols in self._runs:
            t = tab[at:at + len(n)]
            at += len(n)
            for name, v in (("kind", kind), ("k", k), ("n", n), ("dx", dx), ("dy", dy), ("dz", dz), ("n_segs", 1)):
                t[name] = v
            t["col"][:, :cols.shape[1]] = cols
        seg_arr = (ctypes.c_int64 * 1)(0)
        if self._classes is not None:
            tab["n_segs"], tab["seg_index"] = self._classes[:2]
            seg_arr = (ctypes.c_int64 * len(self._classes[2]))(*self._classes[2].tolist())
        return inst_arr, seg_arr

    def arena(self, device, stream):
        return self.device_arena, None

    def point_offsets(self) -> np.ndarray:
        n = np.concatenate([np.zeros(0, dtype=np.int64)] + [r[2] for r in self._runs])
        return np.concatenate([[0], np.cumsum(n)])

    def device(self, flags: int = 0, export: bool = False, hints: bool = True):
        return DeviceBatch(self, flags, export, hints)

    def run(self, flags: int = 0, export: bool = False, hints: bool = True):
        with on(_stream()):
            db = self.device(flags, export, hints)
            db.launch()
            return db.results()


# Values that are copied to pinned memory and sent up at a time, so that one piece
# goes up while the next is copied.  The calling thread copies them: where the
# caller's own program keeps all processors busy (NumPy's threads spin on after a
# matrix product), one that waits for helpers, woken or new, waited 4 ms for them.
_PIECE = 1 << 18
# Pieces in use at a time: pinned memory is kept for later calls, so it is bounded
# (64 MB) whatever the columns take.
_PIECES = 32
# Up to so many values go up in one copy, as columns: the host lays out 16,384 in
# 20 us, what two more copies and the kernel that turns rows into columns take.
_SHORT = 1 << 14


class _Pieces:
    """Pinned memory for `total` values, filled piece by piece from its start, or, where
    they are more than _PIECES pieces, by turns: each quarter of it again once the
    copies from it have ended."""

    def __init__(self, total: int, stream) -> None:
        import torch
        self.size = min(total, _PIECES * _PIECE)
        self.memory = torch.empty(self.size, dtype=torch.float64, pin_memory=True)
        self.turns = total > self.size
        self.sent = [None] * 4   # (with turns) the end of the last copies from each quarter
        self.at = 0              # where the next piece starts
        self.stream = stream

    def _begin(self) -> int:
        if self.turns:
            self.at %= self.size
            q, rest = divmod(self.at, self.size // 4)
            if rest == 0 and self.sent[q] is not None:
                self.sent[q].synchronize()
        return self.at

    def _end(self, count: int) -> None:
        import torch
        self.at += _PIECE if self.turns else count
        if self.turns and self.at % (self.size // 4) == 0:
            q = self.at // (self.size // 4) - 1
            if self.sent[q] is None:
                self.sent[q] = torch.cuda.Event()
            self.sent[q].record(self.stream)

    def send(self, parts, dst) -> None:
        """The values of parts (1-D, or rows of a table), one after the other, to dst."""
        memory = self.memory.view(dst.dtype)
        host, scale = memory.numpy(), len(memory) // self.size
        begin = fill = done = 0
        for a in parts:
            if a.ndim > 1 and (a.flags.c_contiguous or a.shape[1] > _PIECE):
                a = np.ascontiguousarray(a).reshape(-1)
            width = 1 if a.ndim == 1 else a.shape[1]
            n, k = len(a), 0
            while k < n:
                if fill == 0:
                    begin = self._begin() * scale
                rows = min(n - k, (_PIECE - fill) // width)
                if rows > 0:
                    to = host[begin + fill:begin + fill + rows * width]
                    if width > 1:
                        to = to.reshape(rows, width)
                    to[...] = a[k:k + rows]
                    k += rows
                    fill += rows * width
                if fill + width > _PIECE:
                    dst[done:done + fill].copy_(memory[begin:begin + fill], non_blocking=True)
                    self._end(fill)
                    done += fill
                    fill = 0
        if fill > 0:
            dst[done:done + fill].copy_(memory[begin:begin + fill], non_blocking=True)
            self._end(fill)


def upload_columns(arrays, device, stream):
    """The values of arrays (columns, or tables of columns) as float64 columns
    in HBM, one after the other; returns (device columns, pinned host memory).
    They go up from pinned host memory, asynchronously on `stream`, while the
    host goes on; a table held row by row is turned into columns on the device."""
    import torch
    blocks = []   # values as they lie in memory (rows of `m`, or column by column), m
    for a in arrays:
        n = len(a)
        m = 1 if a.ndim == 1 else a.shape[1]
        by_column = m == 1 or a.flags.f_contiguous
        blocks.append((a.reshape(n) if m == 1 else a.T if by_column else a, 1 if by_column else m, n * m))
    total = sum(size for _, _, size in blocks)
    with on(stream):
        if total <= _SHORT:
            pinned = torch.empty(total, dtype=torch.float64, pin_memory=True)
            host, at = pinned.numpy(), 0
            for a, m, size in blocks:
                host[at:at + size].reshape(m, -1)[...] = a.reshape(-1) if m == 1 else a.T
                at += size
            return pinned.to(device, non_blocking=True), pinned
        ctx = nat.context()
        d_cols = torch.empty(total, dtype=torch.float64, device=device)
        pieces = _Pieces(total, stream)
        waiting, begin, at = [], 0, 0   # columns that go up together, from `begin` on

        def send_waiting():
            if waiting:
                pieces.send(waiting, d_cols[begin:at])
                waiting.clear()

        for a, m, size in blocks:
            whole = a.dtype in (np.int64, np.int32)   # go up as they are, become doubles there
            if m > 1 or whole:
                send_waiting()
                dst = d_cols[at:at + size]
                up = torch.empty(size, dtype=getattr(torch, a.dtype.name) if whole else torch.float64, device=device)
                pieces.send([a], up)
                if m > 1:
                    rows = up.to(torch.float64)
                    with ctx.lock:
                        ctx.prep_columns(rows.data_ptr(), size // m, m, dst.data_ptr(), stream.cuda_stream)
                else:
                    dst.copy_(up)
                at += size
                begin = at
            else:
                waiting.append(a)
                at += size
        send_waiting()
    return d_cols, pieces.memory


_side_stream = None


def _stream():
    """A dedicated stream at default priority (hipGraph capture needs a
    non-legacy stream)."""
    global _side_stream
    import torch
    if _side_stream is None:
        nat.context()   # says what is missing without a GPU
        _side_stream = torch.cuda.Stream()
    return _side_stream


_entered = threading.local()   # .stream: the stream of this thread's outermost `on`


class on:
    """torch.cuda.stream(stream), which costs 6 us, entered once by nested uses."""

    def __init__(self, stream) -> None:
        self.stream = stream
        self.context = None

    def __enter__(self) -> None:
        import torch
        if getattr(_entered, "stream", None) is not self.stream:
            self.before = getattr(_entered, "stream", None)
            self.context = torch.cuda.stream(self.stream)
            self.context.__enter__()
            _entered.stream = self.stream

    def __exit__(self, *exc) -> None:
        if self.context is not None:
            _entered.stream = self.before
            self.context.__exit__(*exc)


def on_stream(f):
    """f on the dedicated stream."""
    @functools.wraps(f)
    def g(*args, **kwargs):
        with on(_stream()):
            return f(*args, **kwargs)
    return g
