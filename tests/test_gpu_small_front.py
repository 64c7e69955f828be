"""Small selects whose sample, bracket and sweep share a launch, and those
whose sweep is a launch of its own: sizes around the lines between them, lists
longer than a workgroup gathers in LDS, what the sweep reports, several buckets
at once, and one workspace used by both in turn."""
import pytest
import torch

from oracle import select as SEL
from tests.util import same_bits, student_t

pytestmark = pytest.mark.gpu
CHUNK = 1024
# one slab a wave up to 1024 chunks, four beyond; one launch up to 4096 chunks (1024 for chains of arithmetic)
_SIZES = [1, 3, CHUNK * 4, CHUNK * 4 + 1, CHUNK * 1024 - 1, CHUNK * 1024, CHUNK * 1024 + 1, CHUNK * 1040 + 5,
          CHUNK * 4096, CHUNK * 4096 + 1]


def _select(dev, score, k, ws=None):
    from sga_amd import _lib as L
    from sga_amd.selection import read_result
    n = score.numel()
    if ws is None:
        ws = torch.zeros(int(L.raw("sga_select_workspace_bytes", n)), dtype=torch.uint8, device=dev)
    mask = torch.empty(n, dtype=torch.uint8, device=dev)
    res = torch.empty(8, dtype=torch.int32, device=dev)
    sd = score.to(dev)
    L.call("sga_select_topk", L.ptr(sd), n, k, L.TIE_LOWEST_INDEX, L.ptr(mask), L.ptr(res), L.ptr(ws), ws.numel(),
           L.stream())
    return read_result(res), mask.cpu().bool()


def test_select_sizes_on_one_workspace(dev):
    from sga_amd import _lib as L
    ws = torch.zeros(int(L.raw("sga_select_workspace_bytes", max(_SIZES))), dtype=torch.uint8, device=dev)
    for n in _SIZES + _SIZES[::-1]:
        sc = student_t(n, n % 97).abs()
        for k in {max(1, n // 100), max(1, n // 3)} | ({1, n} if n < CHUNK * 1024 else set()):
            want, thresh = SEL.select_topk_flat(sc, k)
            r, mask = _select(dev, sc, k, ws)
            assert (r.n_selected, r.thresh) == (k, thresh) and torch.equal(mask, want), (n, k)


@pytest.mark.parametrize("n", [CHUNK * 64, CHUNK * 1500 + 7, CHUNK * 4200])
def test_a_workgroup_lists_more_than_it_gathers(dev, n):
    """Everything inside the bracket lies in a few chunks."""
    sc = torch.zeros(n)
    block = min(n // 4, 6 * CHUNK)
    sc[n // 2:n // 2 + block] = torch.rand(block, generator=torch.Generator().manual_seed(n)) * 0.01 + 1.0
    for k in (block // 2, block // 3 + 1):
        want, thresh = SEL.select_topk_flat(sc, k)
        r, mask = _select(dev, sc, k)
        assert (r.n_selected, r.thresh) == (k, thresh) and torch.equal(mask, want), k


@pytest.mark.parametrize("n", [5000, CHUNK * 1024, CHUNK * 3000, CHUNK * 4200 + 3])
def test_reports_of_the_sweep(dev, n):
    sc = student_t(n, 3).abs()
    sc[n - 1], sc[n // 2], sc[0] = float("inf"), float("nan"), float("-inf")
    r, _ = _select(dev, sc, max(1, n // 50))
    assert r.nonfinite == 3 and r.negative
    r, _ = _select(dev, student_t(n, 3).abs(), max(1, n // 50))
    assert r.nonfinite == 0 and not r.negative


@pytest.mark.parametrize("score", ["abs_g", "update", "coi"])
@pytest.mark.parametrize("sizes", [(CHUNK * 1024, 70_001), (CHUNK * 1025,), (300_001, 1_200_003, 5000, 2_000_000)])
def test_steps_agree_with_the_radix_passes(dev, sizes, score):
    """Buckets of one call, all in one launch or not, against the select without a sample; the tensors'
    learning rates change between the steps."""
    from sga_amd.fused_step import FusedSparseStep, fused_step_multi
    ends = []
    for fast in (True, False):
        steppers, views, ks = [], [], []
        for b, n in enumerate(sizes):
            cut = n // 3
            segs = [dict(start=0, n=cut, lr=1e-4, b1=0.9, b2=0.95, eps=1e-8, wd=0.1),
                    dict(start=cut, n=n - cut, lr=2e-4, b1=0.8, b2=0.99, eps=1e-6, wd=0.0)]
            gen = torch.Generator().manual_seed(n)
            p, m = (torch.randn(n, generator=gen) * 0.02).to(dev), (torch.randn(n, generator=gen) * 1e-4).to(dev)
            views.append([student_t(n, b).to(dev), torch.zeros(n, device=dev), p, m,
                          torch.full((n,), 1e-6, device=dev)])
            ks.append(max(1, n // 100))
            steppers.append(FusedSparseStep(n, segs, dev, values_dtype=torch.float32, max_k=ks[-1], want_mask=True))
        out = []
        for t in (1, 2):
            for fs in steppers:
                for s in fs.segments:
                    s["lr"] = 1e-4 * t
            if fast:
                packs = fused_step_multi(steppers, *[[v[j] for v in views] for j in range(5)], t, ks=ks, score=score)
            else:
                packs = [fs.step(*v, t, k=k, score=score, fast=False) for fs, v, k in zip(steppers, views, ks)]
            for (idx, val), fs in zip(packs, steppers):
                out += [idx.clone(), val.clone(), fs.mask.clone()]
        ends.append(out + [x for v in views for x in v])
    for a, b in zip(*ends):
        assert torch.equal(a, b) if a.dtype != torch.float32 else same_bits(a, b)


@pytest.mark.parametrize("tensors", [1, 2, 8192, 8193])
@pytest.mark.parametrize("n", [300_001, 9_000_003])
def test_tables_of_many_tensors(dev, n, tensors):
    """The sample looks tensors up among their starts in LDS, up to 8192 of them; the hyper-parameters decide
    what is selected.  Against the select without a sample."""
    from sga_amd.fused_step import FusedSparseStep
    each = n // tensors
    ends = []
    for fast in (True, False):
        segs = [dict(start=t * each, n=each if t + 1 < tensors else n - t * each, lr=1e-4, b1=0.9, b2=0.95,
                     eps=1e-8 * (1 + 50 * (t % 3)), wd=0.1 * (t % 2)) for t in range(tensors)]
        gen = torch.Generator().manual_seed(tensors)
        state = [torch.zeros(n, device=dev), (torch.randn(n, generator=gen) * 0.02).to(dev),
                 (torch.randn(n, generator=gen) * 1e-4).to(dev), torch.full((n,), 1e-8, device=dev)]
        fs = FusedSparseStep(n, segs, dev, values_dtype=torch.float32, max_k=n // 100)
        idx, val = fs.step(student_t(n, 7).to(dev), *state, 3, k=n // 100, score="update", fast=fast)
        ends.append([idx, val, *state])
    for a, b in zip(*ends):
        assert torch.equal(a, b) if a.dtype != torch.float32 else same_bits(a, b)


# a workgroup's sixteen chunks reserve by fours: the whole list in one of them, over its parts and those of its neighbour
@pytest.mark.parametrize("chunks", [1025, 1031, 2500, 4096])
@pytest.mark.parametrize("how", ["ascending", "descending", "piece"])
def test_lists_of_one_workgroup(dev, chunks, how):
    n = CHUNK * chunks - 3
    sc = torch.rand(n, generator=torch.Generator().manual_seed(chunks)).sort(descending=how == "descending").values
    if how == "piece":
        sc = sc[torch.randperm(n, generator=torch.Generator().manual_seed(1))]
        sc[n // 3:n // 3 + n // 60] += 8
    for k in (200, n // 100, n // 10):
        want, thresh = SEL.select_topk_flat(sc, k)
        r, mask = _select(dev, sc, k)
        assert (r.n_selected, r.thresh, r.path) == (k, thresh, 1) and torch.equal(mask, want), k
