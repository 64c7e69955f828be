"""Workspaces are the caller's and nobody clears them: selects and fused steps
whose workspace holds anything (ones, set bits, odd numbers as a launch might
carry, noise), reused across sizes and kinds of calls."""
import pytest
import torch

from oracle import select as SEL
from tests.util import same_bits, student_t

pytestmark = pytest.mark.gpu

_FILLS = ("ones", "bits", "odd", "noise")


def _dirty(ws, how, seed=0):
    words = ws[:ws.numel() // 4 * 4].view(torch.int32)
    if how == "ones":
        words.fill_(1)
    elif how == "bits":
        words.fill_(-1)
    elif how == "odd":
        words.copy_(torch.arange(words.numel(), dtype=torch.int32, device=ws.device) * 2 + 1)
    else:
        gen = torch.Generator(device=ws.device).manual_seed(seed)
        words.random_(-2 ** 31, 2 ** 31, generator=gen)


# below 2^20 (the sample lies in the candidate list), the sweep's one and four chunks a workgroup, large
_SIZES = [5, 4097, 300_001, 2_200_001, 9_000_003]


@pytest.mark.parametrize("how", _FILLS)
def test_selects_share_one_dirty_workspace(dev, how):
    from sga_amd import _lib as L
    from sga_amd.selection import read_result
    ws = torch.empty(int(L.raw("sga_select_workspace_bytes", max(_SIZES))), dtype=torch.uint8, device=dev)
    for turn, n in enumerate(_SIZES + _SIZES[::-1]):
        sc = student_t(n, n % 89).abs()
        k = max(1, n // 100)
        want, thresh = SEL.select_topk_flat(sc, k)
        if turn % 2 == 0:
            _dirty(ws, how, turn)
        sd = sc.to(dev)
        mask = torch.empty(n, dtype=torch.uint8, device=dev)
        res = torch.empty(8, dtype=torch.int32, device=dev)
        L.call("sga_select_topk", L.ptr(sd), n, k, L.TIE_LOWEST_INDEX, L.ptr(mask), L.ptr(res), L.ptr(ws), ws.numel(),
               L.stream())
        r = read_result(res)
        assert (r.status, r.n_selected, r.thresh) == (0, k, thresh), (n, vars(r))
        assert torch.equal(mask.cpu().bool(), want), n


@pytest.mark.parametrize("how", _FILLS)
@pytest.mark.parametrize("score", ["abs_g", "update"])
@pytest.mark.parametrize("n", _SIZES[1:])
def test_fused_steps_on_dirty_workspaces(dev, n, score, how):
    """Every output as on cleared workspaces, which the other tests compare with the oracle."""
    from sga_amd.fused_step import FusedSparseStep
    segs = [dict(start=0, n=n - 1000, lr=1e-4, b1=0.9, b2=0.95, eps=1e-8, wd=0.1),
            dict(start=n - 1000, n=1000, lr=2e-4, b1=0.8, b2=0.99, eps=1e-6, wd=0.0)]
    gen = torch.Generator().manual_seed(n)
    p = (torch.randn(n, generator=gen) * 0.02).to(dev)
    gs = [student_t(n, s).to(torch.bfloat16).to(dev) for s in (1, 2)]
    ends = []
    for single in (False, True):
        for fill in (None, how):
            fs = FusedSparseStep(n, segs, dev, values_dtype=torch.bfloat16, want_mask=True)
            cur = [torch.zeros(n, device=dev), p.clone(), torch.zeros(n, device=dev), torch.zeros(n, device=dev)]
            nxt = [torch.empty_like(p) for _ in range(4)]
            out = []
            for t, g in enumerate(gs):
                for ws in (fs.ws, fs._single_sweep_ws()) if single else (fs.ws,):
                    ws.zero_() if fill is None else _dirty(ws, fill, t)
                if single:
                    idx, vals = fs.step(g, *cur, t + 1, ratio_percent=1.0, score=score, single_sweep=True, out=nxt)
                    cur, nxt = nxt, cur
                else:
                    idx, vals = fs.step(g, *cur, t + 1, ratio_percent=1.0, score=score)
                assert fs.read_result().status == 0
                out += [idx.clone(), vals.clone(), fs.mask.clone()]
            ends.append(out + cur)
    for end in ends[1:]:
        for a, b in zip(ends[0], end):
            assert torch.equal(a, b) if a.dtype != torch.float32 else same_bits(a, b)


@pytest.mark.parametrize("n", _SIZES[2:])
def test_recorded_selects_and_steps(dev, n):
    """A graph repeats its launches' numbers on the same workspace; eager calls and anything
    else may write there between two replays."""
    from sga_amd import _lib as L
    from sga_amd.fused_step import FusedSparseStep
    k = n // 100
    segs = [dict(start=0, n=n, lr=1e-4, b1=0.9, b2=0.95, eps=1e-8, wd=0.1)]
    ws = torch.zeros(int(L.raw("sga_select_workspace_bytes", n)), dtype=torch.uint8, device=dev)
    score, mask = torch.zeros(n, device=dev), torch.empty(n, dtype=torch.uint8, device=dev)
    res = torch.empty(8, dtype=torch.int32, device=dev)
    fs, ref = (FusedSparseStep(n, segs, dev, values_dtype=torch.float32, max_k=k) for _ in range(2))
    g = torch.zeros(n, device=dev)
    p = (torch.randn(n, generator=torch.Generator().manual_seed(n)) * 0.02).to(dev)
    cur, want = ([torch.zeros_like(p), p.clone(), torch.zeros_like(p), torch.zeros_like(p)] for _ in range(2))

    def work(steps, state):
        L.call("sga_select_topk", L.ptr(score), n, k, L.TIE_LOWEST_INDEX, L.ptr(mask), L.ptr(res), L.ptr(ws), ws.numel(),
               L.stream())
        return steps.step(g, *state, 1, k=k)
    score.copy_(student_t(n, 1).abs())
    g.copy_(student_t(n, 2))
    work(fs, [t.clone() for t in cur])                    # every kernel is loaded once
    torch.cuda.synchronize()
    graph = torch.cuda.CUDAGraph()
    with torch.cuda.graph(graph):
        idx, values = work(fs, cur)
    for turn in range(4):
        sc = student_t(n, 10 + turn).abs()
        score.copy_(sc)
        g.copy_(student_t(n, 20 + turn))
        if turn >= 2:
            _dirty(ws, _FILLS[turn], turn)
            _dirty(fs.ws, _FILLS[turn], turn)
        graph.replay()
        torch.cuda.synchronize()
        expect, _ = SEL.select_topk_flat(sc, k)
        assert torch.equal(mask.cpu().bool(), expect), turn
        mask.zero_()
        i2, v2 = work(ref, want)                          # eager, on the same select workspace
        assert torch.equal(mask.cpu().bool(), expect) and torch.equal(idx, i2) and same_bits(values, v2), turn
        assert all(same_bits(a, b) for a, b in zip(cur, want)), turn
