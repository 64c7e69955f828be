"""Device tables of per-tensor hyper-parameters, laid out once per bucket or
shard; a step rewrites the learning rates and the bias corrections
(``sga_segments_refresh``: the values travel in the kernel arguments, nothing
is staged or waited for), and the whole table only where its rows changed."""
import ctypes as C
from operator import index, itemgetter

import numpy as np
import torch

from . import _lib as L


class ReplaySegment(C.Structure):
    """struct sga_replay_segment"""
    _fields_ = [("start", C.c_int64), ("n", C.c_int64), ("lr", C.c_double), ("wd", C.c_double),
                ("beta1", C.c_float), ("om1", C.c_float), ("beta2", C.c_float),
                ("om2", C.c_float), ("eps", C.c_float), ("bc1", C.c_float), ("bc2", C.c_float),
                ("wdf", C.c_float)]


_HYPER = itemgetter("b1", "b2", "eps", "wd")
_BETAS = itemgetter("b1", "b2")
_SEGMENT, _REPLAY_SEGMENT = np.dtype(L.Segment), np.dtype(ReplaySegment)


def _host_table(dtype, rows, start):
    t = np.zeros(len(rows), dtype=dtype)
    t["start"], t["n"] = [index(r[start]) for r in rows], [index(r["n"]) for r in rows]
    for name, values in (("beta1", [r["b1"] for r in rows]), ("om1", [1.0 - r["b1"] for r in rows]),
                         ("beta2", [r["b2"] for r in rows]), ("om2", [1.0 - r["b2"] for r in rows]),
                         ("eps", [r["eps"] for r in rows])):
        t[name] = list(map(L.f32, values))
    if dtype is _REPLAY_SEGMENT:
        t["wd"] = [float(r["wd"]) for r in rows]
        t["wdf"] = [L.f32(r["wd"]) for r in rows]
    else:
        t["wd"] = [L.f32(r["wd"]) for r in rows]
    return torch.from_numpy(t.view(np.uint8))


class SegmentTable:
    """``rows``: dicts with ``n, b1, b2, eps, wd`` and the first coordinate under
    ``start``.  ``segs`` / ``rsegs`` are the device tables (``sga_segment`` /
    ``sga_replay_segment``) that were asked for."""

    def __init__(self, rows, device, start="start", segs=True, rsegs=False):
        self.count = len(rows)
        self._start = start
        self.segs = _host_table(_SEGMENT, rows, start).to(device) if segs else None
        self.rsegs = _host_table(_REPLAY_SEGMENT, rows, start).to(device) if rsegs else None
        self._lr, self._bc1, self._bc2 = (np.zeros(self.count, dtype=d) for d in ("f8", "f4", "f4"))
        # (segs, rsegs, rows, lr, bc1, bc2): what sga_segments_refresh and sga_replay_begin take
        self.args = (None if self.segs is None else self.segs.data_ptr(),
                     None if self.rsegs is None else self.rsegs.data_ptr(), self.count,
                     self._lr.ctypes.data, self._bc1.ctypes.data, self._bc2.ctypes.data)
        self.cols = L.SegmentCols(*self.args[3:])       # what the fused steps take along
        self._hyper = list(map(_HYPER, rows))
        self._betas = self._last_lr = None
        self.follow_betas(rows)

    def follow_betas(self, rows):
        """Bias corrections are those of the betas that ``rows`` hold now; rows of equal
        betas share them."""
        betas = list(map(_BETAS, rows))
        if betas == self._betas:
            return
        self._betas, groups = betas, {}
        for i, b in enumerate(betas):
            groups.setdefault(b, []).append(i)
        self._groups = [(b, slice(None) if len(groups) == 1 else np.array(at)) for b, at in groups.items()]

    def follow(self, rows):
        """Takes over the betas, eps and weight decay that ``rows`` hold now (4 us
        for 50 rows that did not change; the copy of changed ones waits)."""
        hyper = list(map(_HYPER, rows))
        if hyper == self._hyper:
            return
        for t, dtype in ((self.segs, _SEGMENT), (self.rsegs, _REPLAY_SEGMENT)):
            if t is not None:
                t.copy_(_host_table(dtype, rows, self._start))
        self._hyper = hyper
        self.follow_betas(rows)

    def take(self, lr, count, bias_correction=True):
        """Learning rates (one number, or one per row) and the bias corrections of
        step ``count`` into the host columns, for a call that carries ``args``."""
        lr = list(map(float, lr)) if isinstance(lr, list) else float(lr)   # the caller may change its list
        if lr != self._last_lr:
            self._lr[:] = self._last_lr = lr
        for (b1, b2), at in self._groups:
            self._bc1[at] = float(1.0 - b1 ** count) if bias_correction else 1.0
            self._bc2[at] = float(1.0 - b2 ** count) if bias_correction else 1.0

    def refresh(self, lr, count, bias_correction=True):
        """The same into the device tables, on the current stream."""
        self.take(lr, count, bias_correction)
        L.call("sga_segments_refresh", *self.args, L.stream())
