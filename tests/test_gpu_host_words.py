"""Results that kernels write into words of the host's while it waits: every
value arrives, also those that look like a word that has not."""
import math
import struct

import pytest
import torch

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("bits", [0xFFFFFFFF, 0x7FC00000, 0xFF800000, 0x7F7FFFFF, 0x00000001])
def test_norms_of_any_value_arrive(dev, bits):
    from sga_amd.kernels import compact_norm, compact_norm_sq_contribution
    x = torch.full((5000,), 0.5)
    x.view(torch.int32)[1234] = bits - (1 << 32) if bits >= 1 << 31 else bits
    total = torch.zeros(1, device=dev)
    compact_norm_sq_contribution(x.to(dev), total)
    want, got = total.cpu().sqrt().item(), compact_norm([x.to(dev)])
    assert math.isnan(got) if math.isnan(want) else got == want


@pytest.mark.parametrize("sizes", [(1,), (0, 3), (1024, 0, 1025), (4099, 70_001, 1_000_003)])
def test_norms_of_several_arrays(dev, sizes):
    """Bit for bit the sum that one contribution after the other gives; its root is rounded once."""
    from sga_amd.kernels import compact_norm, compact_norm_sq_contribution
    gen = torch.Generator().manual_seed(sum(sizes))
    arrays = [torch.randn(s, generator=gen).to(dev) for s in sizes]
    total = torch.zeros(1, device=dev)
    for a in arrays:
        compact_norm_sq_contribution(a, total)
    assert struct.pack("<f", compact_norm(arrays)) == struct.pack("<f", total.cpu().sqrt().item())
    assert compact_norm([torch.empty(0, device=dev)]) == 0.0


def test_words_behind_a_long_queue(dev):
    """Nothing arrives for longer than the host looks: it waits for the stream then."""
    from sga_amd.replay import select_topk_flat
    score = torch.rand(300_001, generator=torch.Generator().manual_seed(1)).to(dev)
    big = torch.empty(1 << 28, device=dev)
    torch.cuda.synchronize()
    for _ in range(150):                          # some 40 ms of fills
        big.zero_()
    mask, thresh = select_topk_flat(score, 3000)
    assert int(mask.sum()) == 3000 and thresh == score.topk(3000).values[-1].item()


def test_selects_in_a_row_keep_their_masks(dev):
    """Each call's mask and threshold belong together, however many calls follow."""
    from sga_amd.replay import select_topk_flat
    scores = [torch.rand(n, generator=torch.Generator().manual_seed(n)).to(dev) for n in (5, 70_001, 3_000_017, 12_000_001)]
    got = [select_topk_flat(s, max(1, s.numel() // 50)) for s in scores for _ in range(3)]
    for i, (mask, thresh) in enumerate(got):
        s = scores[i // 3]
        assert torch.equal(mask, s >= thresh) or int(mask.sum()) == max(1, s.numel() // 50)
        assert not bool((mask & (s < thresh)).any()) and not bool((~mask & (s > thresh)).any())


@pytest.mark.parametrize("adams", [False, True])
def test_sums_whose_low_half_has_all_bits_set(dev, adams):
    """Squares of whole numbers that add up to 2^53 - 1, the double 0x433FFFFFFFFFFFFF: every partial sum is
    exact, in any order."""
    from sga_amd.replay_dense import DenseReplay
    left, values = 2 ** 53 - 1, []
    while left:
        values.append(min(math.isqrt(left), 2 ** 24))
        left -= values[-1] ** 2
    assert struct.pack(">d", float(sum(x * x for x in values))).hex() == "433fffffffffffff"
    n = 3 * len(values) + 1000
    g = torch.zeros(n)
    g[torch.arange(len(values)) * 3] = torch.tensor(values, dtype=torch.float32)
    w, m, v = torch.zeros(n, device=dev), torch.zeros(n, device=dev), torch.full((n,), 1.0, device=dev)
    rep = DenseReplay([dict(a=0, n=n, b1=0.9, b2=0.95, eps=1e-8, wd=0.0, group=0)], w, m, v, 3,
                      "adams" if adams else "adamw")
    for t in range(2):
        rep.step(t, g.to(dev), {"lr": [1e-3], "clip_grad": 0.0})
    assert [r["recon_grad_norm"] for r in rep.recon_steps] == [math.sqrt(2.0 ** 53 - 1)] * 2


@pytest.mark.parametrize("n", [5000, 3_000_017, 12_000_001, 200_000_003])
def test_a_select_returns_behind_its_mask(dev, n, monkeypatch):
    """Mask and threshold are there when the call returns: on any stream, without an event."""
    from types import SimpleNamespace
    from sga_amd import config
    from sga_amd.replay import select_topk_flat
    from sga_amd.selection import TopkSelection, select_masks_histogram
    monkeypatch.setattr(config, "_ARGS", SimpleNamespace(sga_selection_method="histogram",
                                                         sga_selection_ratio_percent=2.0))
    score = torch.rand(n, generator=torch.Generator(device=dev).manual_seed(n), device=dev)
    views, k = [score[:n // 2], score[n // 2:]], int(round(n * 0.02))
    plugin, other = TopkSelection(), torch.cuda.Stream()
    ties = int((score >= score.topk(k).values[-1]).sum())
    for call in (lambda: [select_topk_flat(score, k)[0]], lambda: select_masks_histogram(views, k)[1],
                 lambda: plugin.select(SimpleNamespace(grad_views=[score]))):
        torch.cuda.synchronize()
        with torch.cuda.stream(other):
            torch.zeros(1, device=dev)                # the other stream is there
        masks = call()
        with torch.cuda.stream(other):
            on = sum(int(m.sum(dtype=torch.int64)) for m in masks)
        assert on in (k, ties)                    # of the scores at the threshold as many as make k, or all


@pytest.mark.parametrize("wide", [False, True])
def test_words_given_up_early_stay_out_of_the_pool(dev, wide):
    """Whoever stops waiting (an interrupt, an error) leaves a kernel behind that has yet to write: nobody
    else's words lie there before it has; afterwards the memory is used again."""
    from sga_amd import _lib as L
    big = torch.empty(1 << 28, device=dev)
    x, partials = torch.ones(5000, device=dev), torch.empty(2048, device=dev)
    grad, idx, values = torch.ones(9, device=dev), torch.arange(5, dtype=torch.int32, device=dev), torch.empty(5, device=dev)

    def launch():
        w = L.words(1, wide)
        if wide:
            L.call("sga_pack_selected_split", L.ptr(grad), L.ptr(idx), L.ptr(values), L.SGA_F32, 1.0, 5, 9, 3, L.ptr(w),
                   L.stream())
        else:
            L.call("sga_compact_norm_sq_from", L.ptr(x), 5000, L.ptr(partials), None, L.ptr(w), L.stream())
        return w
    assert L.arrived(launch()) == ((3,) if wide else (0x459C4000,))
    torch.cuda.synchronize()
    for _ in range(150):                          # some 40 ms of fills
        big.zero_()
    given_up = [launch() for _ in range(4)]
    there = {w.data_ptr() for w in given_up}
    del given_up
    assert not torch.cuda.current_stream().query()
    later = [L.words(1, wide) for _ in range(40)]
    assert not there & {w.data_ptr() for w in later}
    torch.cuda.synchronize()
    assert all(w.item() == -1 for w in later)
    del later
    torch.cuda.synchronize()
    seen = set()
    for _ in range(300):
        w = launch()
        L.arrived(w)
        seen.add(w.data_ptr())
        del w
    assert len(seen) < 100


@pytest.mark.parametrize("call", ["index", "mask", "norm"])
def test_an_interrupted_wait(dev, call, monkeypatch):
    """The next call has its own words, whatever the one before has left on the stream."""
    from sga_amd import _lib as L
    from sga_amd.backends import index_layout_pack, mask_layout_pack
    from sga_amd.kernels import compact_norm
    n = 100_000
    mask = torch.zeros(n, dtype=torch.uint8, device=dev)
    mask[1::7] = 1
    idx, grad = mask.nonzero().view(-1).to(torch.int32), torch.ones(n, device=dev)
    values, big = torch.empty(idx.numel(), device=dev), torch.empty(1 << 28, device=dev)
    run = {"index": lambda m: index_layout_pack(grad, idx[:m], values)[0][1], "mask": lambda m: mask_layout_pack(
        grad, mask * (m > 0))[1].numel(), "norm": lambda m: compact_norm([grad[:m]])}[call]
    want = {"index": lambda m: min(m, int((idx < n // 2).sum())), "mask": lambda m: idx.numel(),
            "norm": lambda m: float(torch.tensor(float(m)).sqrt())}[call]
    run(10)
    torch.cuda.synchronize()
    arrived = L.arrived

    def interrupted(t):
        raise KeyboardInterrupt
    for _ in range(150):
        big.zero_()
    monkeypatch.setattr(L, "arrived", interrupted)
    for _ in range(4):
        with pytest.raises(KeyboardInterrupt):
            run(77)
    monkeypatch.setattr(L, "arrived", arrived)
    grad.fill_(1.0)
    for m in (500, 9000, 3):
        assert run(m) == want(m)


def test_results_without_the_native_host_side(dev, monkeypatch):
    """Selects, compaction, the layouts, the compact norm and the dense replay need libsga_hip.so alone."""
    from sga_amd import _lib as L
    from sga_amd.backends import index_layout_pack, mask_layout_pack
    from sga_amd.kernels import compact_norm
    from sga_amd.replay import select_topk_flat
    from sga_amd.replay_dense import DenseReplay
    from sga_amd.selection import select_masks_histogram
    from sga_amd.support import compact_mask_u8
    n = 70_001
    score = torch.rand(n, generator=torch.Generator().manual_seed(3)).to(dev)

    def results():
        mask, thresh = select_topk_flat(score, 700)
        views = [score[:30_000], score[30_000:]]
        t2, masks = select_masks_histogram(views, 700)
        idx, before = compact_mask_u8(mask.view(torch.uint8), step=n // 3, cuts=2)
        grad, values = score.clone(), torch.empty(700, device=dev)
        bounds = index_layout_pack(grad, idx, values)
        payloads, _ = mask_layout_pack(score, mask.view(torch.uint8))
        rep = DenseReplay([dict(a=0, n=n, b1=0.9, b2=0.95, eps=1e-8, wd=0.0, group=0)], score, score * 0.1,
                          score * score, 3)
        rep.step(0, score, {"lr": [1e-3], "clip_grad": 0.0})
        return ([mask, idx, grad, values, rep.w, *masks, *payloads],
                [thresh, t2, before, bounds, compact_norm([score, values]), rep.recon_steps[0]["recon_grad_norm"]])
    tensors, numbers = results()

    def missing():
        raise RuntimeError("sga_amd/_host.so is missing")
    monkeypatch.setattr(L, "host", missing)
    monkeypatch.setattr(L, "_host_loads", None)
    t2, n2 = results()
    assert all(torch.equal(a, b) for a, b in zip(tensors, t2)) and numbers[:4] == n2[:4]
    # the root of the norm is the host's or the device's
    assert numbers[5] == n2[5] and abs(numbers[4] - n2[4]) <= 2.0 ** -22 * numbers[4]


def test_a_recorded_graph_keeps_no_words_of_the_host(dev):
    from sga_amd import _lib as L
    grad, idx, values = torch.ones(9, device=dev), torch.arange(5, dtype=torch.int32, device=dev), torch.empty(5, device=dev)
    L.arrived(L.words(0, True))
    graph = torch.cuda.CUDAGraph()
    with torch.cuda.graph(graph):
        below = L.words(1, wide=True)
        L.call("sga_pack_selected_split", L.ptr(grad), L.ptr(idx), L.ptr(values), L.SGA_F32, 1.0, 5, 9, 3, L.ptr(below),
               L.stream())
    assert below.is_cuda
    for _ in range(3):
        below.fill_(-1)
        graph.replay()
        torch.cuda.synchronize()
        assert L.arrived(below) == [3]
    assert not L.words(1).is_cuda


@pytest.mark.parametrize("n", [1, 8, 63, 64])
def test_words_to_host(dev, n):
    from sga_amd import _lib as L
    src = torch.randint(-2 ** 31, 2 ** 31 - 1, (n + 1,), dtype=torch.int32, device=dev)
    src[src == -1] = 0
    for at in (0, 1):
        words = L.words(n)
        L.call("sga_words_to_host", L.ptr(src[at:]), n, L.ptr(words), L.stream())
        assert [w & 0xFFFFFFFF for w in src[at:at + n].tolist()] == list(L.arrived(words))
    for bad in (0, 65, -1):
        with pytest.raises(RuntimeError, match="bad argument"):
            L.call("sga_words_to_host", L.ptr(src), bad, L.ptr(words), L.stream())
