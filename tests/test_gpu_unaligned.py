"""Quads at any element's address: views that begin 1, 2 or 3 elements past an
aligned one give the bits that aligned copies of the same data give, at the
edges of a chunk (1024), a workgroup's span (4096) and behind many of them."""
import pytest
import torch

from tests.util import same_bits, student_t

pytestmark = pytest.mark.gpu

SIZES = [1023, 1025, 4097, 300_003]


def _shifted(t, off):
    buf = torch.zeros(t.numel() + 8, dtype=t.dtype, device=t.device)
    view = buf[off:off + t.numel()]
    view.copy_(t)
    return view, buf


def _state(n, dev, grad):
    gen = torch.Generator().manual_seed(n)
    g = student_t(n, 1).to(dev).to(grad)
    r, p, m = (torch.randn(n, generator=gen).mul_(s).to(dev) for s in (3e-4, 0.02, 1e-4))
    v = torch.rand(n, generator=gen).add_(0.05).mul_(1e-6).to(dev)
    return g, r, p, m, v


@pytest.mark.parametrize("n", SIZES)
@pytest.mark.parametrize("off", [1, 2, 3])
@pytest.mark.parametrize("grad", [torch.bfloat16, torch.float32])
@pytest.mark.parametrize("score", ["abs_g", "update"])
def test_fused_step(dev, n, off, grad, score):
    from sga_amd.fused_step import FusedSparseStep
    from sga_amd.shapes import segments_for
    segs, _ = segments_for([("a", n // 3), ("b", n - n // 3)])
    k = n // 50
    outs = []
    for shift in (0, off):
        st = [_shifted(t, shift) for t in _state(n, dev, grad)]
        fs = FusedSparseStep(n, segs, dev, values_dtype=torch.bfloat16, max_k=k, want_mask=True)
        idx, val = fs.step(*(t for t, _ in st), 7, k=k, score=score)
        outs.append([idx.clone(), val.clone(), fs.mask.clone()] + [t.clone() for t, _ in st[1:]])
        for (view, buf) in st:                       # nothing beside the view is written
            assert not buf[:shift].any() and not buf[shift + n:].any()
    for a, b in zip(*outs):
        assert torch.equal(a, b) if not a.is_floating_point() else same_bits(a.float(), b.float())


@pytest.mark.parametrize("n", SIZES + [9_000_001])
@pytest.mark.parametrize("off", [1, 2, 3])
def test_select_and_compaction(dev, n, off):
    from sga_amd.replay import select_topk_flat
    from sga_amd.support import compact_mask_u8
    sc = student_t(n, 9).abs().to(dev)
    view, _ = _shifted(sc, off)
    (m0, t0), (m1, t1) = select_topk_flat(sc, n // 40), select_topk_flat(view, n // 40)
    assert torch.equal(m0, m1) and float(t0) == float(t1)
    mv, _ = _shifted(m0.view(torch.uint8), off)
    assert torch.equal(compact_mask_u8(mv), m0.nonzero()[:, 0].to(torch.int32))


# the large buckets' sweeps: bit planes and settlement (a score that reads every array), and the single
# sweep that writes the new state beside the old
@pytest.mark.parametrize("single_sweep", [False, True])
@pytest.mark.parametrize("off,grad", [(1, torch.bfloat16), (3, torch.float32)])
def test_large_fused_step(dev, off, grad, single_sweep):
    from sga_amd.fused_step import FusedSparseStep
    from sga_amd.shapes import segments_for
    n = 8192 * 1024 + 1027
    segs, _ = segments_for([("a", n // 3), ("b", n - n // 3)])
    k = n // 50
    outs = []
    for shift in (0, off):
        st = [_shifted(t, shift) for t in _state(n, dev, grad)]
        new = [_shifted(torch.zeros(n, device=dev), shift) for _ in range(4)] if single_sweep else st[1:]
        fs = FusedSparseStep(n, segs, dev, values_dtype=torch.bfloat16, max_k=k, want_mask=True)
        knobs = dict(single_sweep=True, seed=5, out=[t for t, _ in new]) if single_sweep else {}
        idx, val = fs.step(*(t for t, _ in st), 7, k=k, score="update", **knobs)
        outs.append([idx.clone(), val.clone(), fs.mask.clone()] + [t.clone() for t, _ in new])
        for (view, buf) in st + new:                 # nothing beside the view is written
            assert not buf[:shift].any() and not buf[shift + n:].any()
    for a, b in zip(*outs):
        assert torch.equal(a, b) if not a.is_floating_point() else same_bits(a.float(), b.float())
