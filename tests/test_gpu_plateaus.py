"""Plateaus of equal scores around the k-th: the sampled bracket shrinks to the one
key, and the lists of the smaller ones are walked in order all the same."""
import pytest
import torch

from oracle import select as SEL
from tests.util import student_t

pytestmark = pytest.mark.gpu


def _plateau(n, k, above, below):
    """Scores whose ranks k - above .. k + below share one value."""
    sc = student_t(n, n % 83).abs()
    top = torch.topk(sc, k + below).values
    return torch.where((sc >= top[-1]) & (sc <= top[k - above]), top[-1], sc), top[-1]


def _select(dev, sc, k):
    from sga_amd import _lib as L
    from sga_amd.selection import read_result
    n = sc.numel()
    ws = torch.zeros(int(L.raw("sga_select_workspace_bytes", n)), dtype=torch.uint8, device=dev)
    sd = sc.to(dev)
    mask = torch.empty(n, dtype=torch.uint8, device=dev)
    res = torch.empty(8, dtype=torch.int32, device=dev)
    L.call("sga_select_topk", L.ptr(sd), n, k, L.TIE_LOWEST_INDEX, L.ptr(mask), L.ptr(res), L.ptr(ws), ws.numel(),
           L.stream())
    r = read_result(res)
    want, thresh = SEL.select_topk_flat(sc, k)
    assert (r.status, r.n_selected, r.thresh) == (0, k, thresh), vars(r)
    assert torch.equal(mask.cpu().bool(), want)
    return ws[48:56].view(torch.int32).tolist()             # SelState.t_lo, t_hi


# plateaus a little wider than the bracket's ranks in the sample: its ends lie on them, with little of their bin outside
@pytest.mark.parametrize("n,above,below", [(300_001, 0.73, 0.73), (3_000_017, 0.525, 0.525), (8_388_608, 0.525, 0.525),
                                           (20_000_003, 1.0, 1.0)])
def test_the_bracket_shrinks_to_a_plateau(dev, n, above, below):
    k = n // 100
    sc, value = _plateau(n, k, int(above * k), int(below * k))
    lo, hi = _select(dev, sc, k)
    assert (lo, hi) == (int(value.view(torch.int32)), int(value.view(torch.int32)) + 1)


# plateaus inside the bracket, in the part of the list that is read on from memory (beyond 1280 entries a wave)
@pytest.mark.parametrize("n,ratio,f", [(3_000_017, 10, 0.05), (8_388_608, 1, 0.3), (8_388_608, 3, 0.1),
                                       (8_388_608, 10, 0.12)])
def test_plateaus_in_long_lists(dev, n, ratio, f):
    k = n * ratio // 100
    for above, below in ((f / 2, f / 2), (f, 0.001), (0.001, f)):
        _select(dev, _plateau(n, k, int(above * k), max(1, int(below * k)))[0], k)
