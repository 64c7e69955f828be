"""Learning rates and bias corrections that a step takes along: the same bits as with the tables brought up
to date by a launch of their own, whatever path the bucket's select takes: small or large, or by radix passes
(``fast=False``), whose steps bring the table up to date by that launch themselves."""
import pytest
import torch

pytestmark = pytest.mark.gpu


def _bucket(dev, n, tensors, seed):
    from sga_amd.fused_step import FusedSparseStep, k_for
    g = torch.Generator(device=dev).manual_seed(seed)
    cuts = [n * i // tensors for i in range(tensors + 1)]
    segs = [dict(start=a, n=b - a, lr=1e-3, b1=0.9, b2=0.95, eps=1e-8, wd=0.1 * (i % 2))
            for i, (a, b) in enumerate(zip(cuts[:-1], cuts[1:]))]
    state = [torch.randn(n, generator=g, device=dev) * s for s in (3e-4, 0.02, 1e-4)]
    state.append((torch.rand(n, generator=g, device=dev) + 0.05) * 1e-6)
    grads = [(torch.randn(n, generator=g, device=dev) * 1e-3).bfloat16() for _ in range(3)]
    return FusedSparseStep(n, segs, dev, max_k=k_for(n, 1.0), want_mask=True), state, grads


def _run(dev, ahead, n, tensors, rates, score, buckets, fast=True):
    from sga_amd.fused_step import fused_step_multi, k_for
    sets = [_bucket(dev, m, t, 7 + i) for i, (m, t) in enumerate(zip(n, tensors))]
    out = []
    for step in range(1, 4):             # the bias corrections move most in the first steps
        for fs, _state, _grads in sets:
            for i, s in enumerate(fs.segments):
                s["lr"] = 1e-3 * (1 + (i + step) % rates)
            if ahead:
                fs._upload_segments(step)
        gs = [grads[step - 1] for _fs, _state, grads in sets]
        if buckets:
            packs = fused_step_multi([s[0] for s in sets], gs, *zip(*[s[1] for s in sets]), step,
                                     ratio_percent=1.0, score=score, fast=fast)
        else:
            fs, state, _grads = sets[0]
            packs = [fs.step(gs[0], *state, step, k=k_for(n[0], 1.0), score=score, fast=fast)]
        out += [t.clone() for p in packs for t in p]
        out += [t.clone() for fs, state, _grads in sets for t in (*state, fs.mask)]
    return out


# tensors: inside a byte's rows and beyond them; rates: inside the triples' number and beyond
@pytest.mark.parametrize("score", ["abs_g", "update"])
@pytest.mark.parametrize("n,tensors,rates", [(5000, 3, 3), (1_200_001, 480, 4), (1_200_001, 481, 4), (300_000, 40, 11),
                                             (9_000_001, 100, 2)])
def test_columns_by_argument(dev, n, tensors, rates, score):
    ends = [_run(dev, ahead, [n], [tensors], rates, score, False, fast) for fast in (True, False) for ahead in (False, True)]
    assert all(torch.equal(x, y) for end in ends[1:] for x, y in zip(ends[0], end))


@pytest.mark.parametrize("n,tensors", [((4097, 70_001, 1, 1_500_000), (5, 60, 1, 200)),
                                       ((200_001,) * 10, (50,) * 10), ((300_000, 9_000_001, 8_500_000), (7, 9, 400))])
def test_columns_of_several_buckets(dev, n, tensors):
    a = _run(dev, False, n, tensors, 2, "update", True)
    for ahead, fast in ((True, True), (False, False), (True, False)):
        assert all(torch.equal(x, y) for x, y in zip(a, _run(dev, ahead, n, tensors, 2, "update", True, fast)))
    single = [t for i in range(len(n)) for t in _run_one(dev, n, tensors, i)]
    assert all(torch.equal(x, y) for x, y in zip(a[-5 * len(n):], single))


def _run_one(dev, n, tensors, i):
    """State and mask of bucket i after the three steps, by steps of its own."""
    from sga_amd.fused_step import k_for
    fs, state, grads = _bucket(dev, n[i], tensors[i], 7 + i)
    for step in range(1, 4):
        for j, s in enumerate(fs.segments):
            s["lr"] = 1e-3 * (1 + (j + step) % 2)
        fs.step(grads[step - 1], *state, step, k=k_for(n[i], 1.0), score="update")
    return [*state, fs.mask]
