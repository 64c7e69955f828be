"""Dense reference pass of the offline replay on the device
(``dense_replay_dev``, ``sga/replay.py:848-926``): the full-gradient AdamW /
AdamS trajectory from a branch point, the per-coordinate label
``sum_t (lr_t * upd_t)^2``, per-horizon ``||w_d(H) - w0||`` and snapshots of
``w_d``, and the pre-clip reconstruction diagnostics of every step.

State is flat over the shard (one launch per recorded step, per-tensor
hyper-parameters through a segment table) and the snapshots stay resident on
the device, where the sparse arms compare against them.
"""
import math

import torch

from . import _lib as L
from .replay import coef_dense_for
from .segments import SegmentTable
from .trace_io import lr_for_step


def lr_max_abs_diff(gmeta):
    """Largest |lr_g - mean lr| over the recorded groups (``replay.py:260-265``)."""
    lrs = [float(x) for x in gmeta.get("lr", [])]
    if not lrs:
        return 0.0
    mean = sum(lrs) / len(lrs)
    return max(abs(x - mean) for x in lrs)


def lr_by_group(gmeta, entries):
    """``lr_for_step`` of every entry, each group looked up once."""
    groups = [e.get("group") for e in entries]
    of = {g: float(lr_for_step(gmeta, g)) for g in set(groups)}
    return [of[g] for g in groups]


class DenseReplay:
    """Resident dense trajectory over a flat shard; ``entries`` as in
    ``ShardParams`` ({"a", "n", "b1", "b2", "eps", "wd", "group"})."""

    def __init__(self, entries, w0, m0, v0, t0, optimizer="adamw"):
        if optimizer not in ("adamw", "adams"):
            raise ValueError(f"unknown optimizer {optimizer!r}")
        L.require_dev(w0, m0, v0)
        self.entries, self.t0, self.optimizer = entries, t0, optimizer
        self.N = w0.numel()
        self.w0 = w0
        self.w, self.m, self.v = w0.clone(), m0.clone(), v0.clone()
        dev = w0.device
        self.label = torch.zeros(self.N, dtype=torch.float32, device=dev)
        self._partials = torch.empty(int(L.raw("sga_replay_partials")), dtype=torch.float64,
                                     device=dev)
        self._dist = torch.zeros(1, dtype=torch.float64, device=dev)
        self._seg_table = SegmentTable(entries, dev, start="a", segs=False, rsegs=True)
        self.si = 0
        self.den_at, self.snapshots, self.recon_steps = {}, {}, []

    def step(self, gstep, g, gmeta, horizons=()):
        """Commit one recorded step; ``g`` is the flat post-clip gradient
        (bf16 or fp32) on the device."""
        L.require_dev(g)
        L.require_contig(g=g)
        if g.numel() != self.N:
            raise ValueError("gradient length does not match the shard")
        coef_dense, flag = coef_dense_for(gmeta)
        count = self.t0 + self.si + 1
        self._seg_table.follow(self.entries)          # callers may change them between steps
        self._seg_table.take(lr_by_group(gmeta, self.entries), count, self.optimizer == "adamw")
        st = L.stream()
        # the fold writes its sum straight into host memory: a step waits for it, and a copy would be
        # one more thing to wait for
        recon2 = L.words(1, wide=True)
        L.call("sga_dense_replay_step_at", L.ptr(g), L.dtype_code(g), L.ptr(self.w), L.ptr(self.m),
               L.ptr(self.v), L.ptr(self.label), self.N, *self._seg_table.args[1:],
               int(self.optimizer == "adams"), float(coef_dense), L.ptr(self._partials),
               L.ptr(recon2), st)
        norm = float(gmeta.get("grad_norm", float("nan")))
        record = {
            "step": gstep, "lr": lr_for_step(gmeta), "lr_max_abs_diff": lr_max_abs_diff(gmeta),
            "grad_norm": norm, "clip_grad": float(gmeta.get("clip_grad", 0.0)),
            "coef_dense": coef_dense, "reconstruct_flag": flag}
        L.arrived(recon2)
        recon = math.sqrt(float(recon2.view(torch.float64).item()))
        record.update(recon_grad_norm=recon, recon_rel_err=((recon - norm) / norm
                                                            if math.isfinite(norm) and norm > 0.0 else None))
        self.recon_steps.append(record)
        self.si += 1
        if self.si in horizons:
            L.call("sga_sq_dist", L.ptr(self.w), 0, L.ptr(self.w0), self.N, L.ptr(self._partials),
                   L.ptr(self._dist), st)
            self.den_at[self.si] = math.sqrt(float(self._dist.item()))
            self.snapshots[self.si] = self.w.clone()

    def label_total(self):
        return float(self.label.sum(dtype=torch.float64).item())


def dense_replay_dev(entries, w0, m0, v0, reader, t0, eff_horizons, optimizer="adamw"):
    """Run the dense pass over a window; ``reader`` yields
    ``(gstep, meta, g_flat)``.  Returns ``(label_total, den_at, recon_steps,
    snapshots, dense)`` with the label left on the device in ``dense.label``."""
    dense = DenseReplay(entries, w0, m0, v0, t0, optimizer)
    for gstep, gmeta, g in reader:
        dense.step(gstep, g, gmeta, eff_horizons)
    return dense.label_total(), dense.den_at, dense.recon_steps, dense.snapshots, dense
