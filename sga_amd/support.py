"""Support helpers of ``sga/support.py`` on MI355X: mask -> sorted int32 idx."""
from typing import Optional

import torch

from . import _lib as L

_GATHER_BUF_CHUNK = 4 << 20   # growth granularity, sga/support.py:29


class IndexPool:
    """Grow-only int32 buffer reused across cycles (``sga/support.py:32-54``)."""

    def __init__(self):
        self.buf: Optional[torch.Tensor] = None

    def get(self, k, device):
        if self.buf is None or self.buf.numel() < k or self.buf.device != device:
            cap = -(-k // _GATHER_BUF_CHUNK) * _GATHER_BUF_CHUNK
            if self.buf is not None and self.buf.device == device:
                cap = max(cap, self.buf.numel())
            self.buf = torch.empty(cap, dtype=torch.int32, device=device)
        return self.buf


def mask_totals(mask_u8, step=0, cuts=0):
    """First half of a compaction: ``(flat uint8 mask, scratch, k, [set bytes before step,
    2 * step, ...])``, with one host read.  The second half is ``sga_mask_list``."""
    n = mask_u8.numel()
    assert n < 2 ** 31, f"int32 support indices assume < 2^31 elements, got {n}"
    L.require_dev(mask_u8)
    mk = mask_u8.reshape(-1)
    L.require_contig(mask_u8=mk)
    if mk.dtype == torch.bool:
        mk = mk.view(torch.uint8)
    if mk.dtype != torch.uint8:
        raise TypeError("compact_mask_u8: uint8/bool mask")
    if n == 0:
        return mk, None, 0, [0] * cuts
    scratch = torch.empty(int(L.raw("sga_mask_list_words", n)), dtype=torch.int32, device=mk.device)
    totals = L.words(1 + cuts, wide=True)
    L.call("sga_mask_totals", L.ptr(mk), n, L.ptr(scratch), step, cuts, L.ptr(totals), L.stream())
    k, *before = L.arrived(totals)
    return mk, scratch, k, before


def compact_mask_u8(mask_u8, pool: Optional[IndexPool] = None, step=0, cuts=0):
    """Ascending int32 positions of the non-zero bytes of ``mask_u8``
    (``sga/support.py:57-99``): one counting sweep, one host read of k (the
    reference syncs on the count too), one ordered fill sweep.  With ``cuts`` the
    same read also brings how many positions lie before ``step``, ``2 * step``, ...:
    returns ``(idx, [that many ints])``."""
    mk, scratch, k, before = mask_totals(mask_u8, step, cuts)
    dev, n = mk.device, mk.numel()
    buf = pool.get(k, dev) if pool is not None and n else torch.empty(
        k, dtype=torch.int32, device=dev)
    if k:
        L.call("sga_mask_list", L.ptr(mk), n, L.ptr(scratch), L.ptr(buf), buf.numel(), None, 1.0,
               None, None, 0, L.stream())
    return (buf[:k], before) if cuts else buf[:k]


def block_idx_from_mask(mask_u8, spans, x):
    """int32 block-start index per x-element block that has ANY set byte, per
    span; blocks tile each span from its start, the tail block may be short
    (``sga/support.py:102-142``).  With x == 1 equals ``compact_mask_u8``."""
    assert mask_u8.numel() < 2 ** 31, (
        f"int32 block-start indices assume < 2^31 elements, got {mask_u8.numel()}")
    L.require_dev(mask_u8)
    mk = mask_u8.reshape(-1)
    if mk.dtype == torch.bool:
        mk = mk.view(torch.uint8)
    dev = mk.device
    prev_end, counts = 0, []
    for start, end in spans:
        assert start >= prev_end, (
            f"spans must be ascending and non-overlapping, got span starting at {start} "
            f"after one ending at {prev_end}")
        prev_end = end
        counts.append(-(-(end - start) // x))
    total = sum(counts)
    if total == 0:
        return torch.empty(0, dtype=torch.int32, device=dev)
    any_b = torch.empty(total, dtype=torch.uint8, device=dev)
    st = L.stream()
    off = 0
    for (start, end), nb in zip(spans, counts):
        if nb:
            L.call("sga_block_any", L.ptr(mk[start:end]), end - start, x,
                   L.ptr(any_b[off:off + nb]), st)
        off += nb
    ordinal = compact_mask_u8(any_b).long()        # selected block ordinals, ascending
    if ordinal.numel() == 0:
        return torch.empty(0, dtype=torch.int32, device=dev)
    first = torch.tensor([0] + list(torch.tensor(counts).cumsum(0)[:-1]), device=dev)
    starts = torch.tensor([s for s, _ in spans], device=dev)
    owner = torch.searchsorted(first, ordinal, right=True) - 1
    return ((ordinal - first[owner]) * x + starts[owner]).to(torch.int32)
