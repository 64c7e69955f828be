"""Mask compaction by 16-byte loads and the slice ends that come with its count, at the edges of
a lane's bytes, a chunk, a workgroup's chunks and the scan's one workgroup, against torch on the CPU."""
import pytest
import torch

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("n", [1, 15, 16, 17, 1023, 1025, 16_385, 100_003, 4096 * 1024, 4096 * 1024 + 1])
@pytest.mark.parametrize("at", [0, 3])
def test_positions_and_slice_ends(dev, n, at):
    from sga_amd.support import compact_mask_u8
    gen = torch.Generator().manual_seed(n)
    buf = torch.zeros(n + at, dtype=torch.uint8)
    buf[at:] = torch.where(torch.rand(n, generator=gen) < 0.05, torch.randint(1, 256, (n,), generator=gen), 0)
    buf[-1] = 255
    on = buf[at:].nonzero().view(-1).to(torch.int32)
    for cuts in (0, 1, 2, 6):
        step = n // (cuts + 1)
        out = compact_mask_u8(buf.to(dev)[at:], step=step, cuts=cuts)
        idx, before = out if cuts else (out, [])
        assert torch.equal(idx.cpu(), on)
        assert before == [int((on < (j + 1) * step).sum()) for j in range(cuts)]


@pytest.mark.parametrize("n", [3, 50_001])
@pytest.mark.parametrize("slices", [1, 2, 5])
def test_mask_layout_slices(dev, n, slices):
    from sga_amd.backends import mask_layout_pack
    gen = torch.Generator().manual_seed(n)
    mask = (torch.rand(n, generator=gen) < 0.1).to(torch.uint8)
    mask[n // 2] = 1
    grad = torch.randn(n, generator=gen)
    payloads, idx = mask_layout_pack(grad.to(dev), mask.to(dev), factor=0.5, slices=slices)
    base = n // slices if slices > 1 else n
    ends = [i * base for i in range(slices)] + [n]
    assert torch.equal(idx.cpu(), mask.nonzero().view(-1).to(torch.int32))
    assert len(payloads) == slices
    for p, a, b in zip(payloads, ends[:-1], ends[1:]):
        assert torch.equal(p.cpu(), grad[a:b][mask[a:b].bool()] * 0.5)


# cuts far past the end: j * step must not wrap around into the list (2 * 2^62 would)
@pytest.mark.parametrize("n", [0, 1, 5000])
@pytest.mark.parametrize("step", [2 ** 31, 2 ** 62, 2 ** 63 - 1])
def test_steps_past_the_end(dev, n, step):
    from sga_amd import _lib as L
    mask = torch.ones(n, dtype=torch.uint8, device=dev)
    counts = torch.empty(int(L.raw("sga_mask_chunks", n)) + 8, dtype=torch.int32, device=dev)
    totals = torch.full((6,), -1, dtype=torch.int64, device=dev)
    L.call("sga_mask_count_cuts", L.ptr(mask), n, L.ptr(counts), step, 5, L.ptr(totals), L.stream())
    assert totals.tolist() == [n] * 6


# chunks just below, at and above the density from which their positions are staged, all set, and lists shorter
# than the mask has bytes
@pytest.mark.parametrize("at", [0, 3])
@pytest.mark.parametrize("counts", [[159, 160, 161, 0, 1024], [1024] * 9, [1, 1023, 1024, 17, 500, 160]])
def test_dense_chunks_and_short_lists(dev, counts, at):
    from sga_amd import _lib as L
    gen = torch.Generator().manual_seed(sum(counts))
    n = 1024 * len(counts) - 5 * (counts[-1] < 1000)
    mask = torch.zeros(1024 * len(counts) + at, dtype=torch.uint8)
    for c, k in enumerate(counts):
        mask[at + 1024 * c:at + 1024 * (c + 1)][torch.randperm(1019 if k < 1000 else 1024, generator=gen)[:k]] = 1 + c
    on = mask[at:at + n].nonzero().view(-1).to(torch.int32)
    md = mask.to(dev)[at:at + n]
    work = torch.empty(int(L.raw("sga_mask_chunks", n)), dtype=torch.int32, device=dev)
    total = torch.empty(1, dtype=torch.int64, device=dev)
    L.call("sga_mask_count", L.ptr(md), n, L.ptr(work), L.ptr(total), L.stream())
    k = on.numel()
    assert total.item() == k
    for cap in sorted({1, 3, 159, 160, 163, k // 2, k - 1, k, k + 7}):
        idx = torch.full((max(cap, k) + 8,), -7, dtype=torch.int32, device=dev)
        L.call("sga_mask_fill", L.ptr(md), n, L.ptr(work), L.ptr(idx), cap, L.stream())
        got, put = idx.cpu(), min(cap, k)
        assert torch.equal(got[:put], on[:put]) and bool((got[put:] == -7).all()), cap
