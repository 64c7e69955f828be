"""Ties at the threshold of a large bucket, more than the settlement ranks by itself: the ordered
prefixes and the ties that they grant are items of one launch."""
import pytest
import torch

from tests.util import student_t

pytestmark = pytest.mark.gpu


def _expected(sc, k):
    """(mask, threshold) with the lowest-index ties, by sorting on the device."""
    t = torch.sort(sc, descending=True)[0][k - 1]
    mask = sc > t
    ties = (sc == t).nonzero().reshape(-1)
    need = k - int(mask.sum())
    mask[ties[:need]] = True
    return mask, float(t), need, ties.numel()


# both sides of the 4096 ties that the settlement ranks, the last chunk whole and ragged
@pytest.mark.parametrize("n", [8192 * 1024 + 1, 8192 * 1024 + 1024 * 4096 - 1, 20_971_520])
@pytest.mark.parametrize("ties", [4096, 4097, 30_000])
def test_ties_beyond_the_settlement(dev, n, ties):
    from sga_amd import _lib as L
    from sga_amd.selection import read_result, select_exact_device
    sc = student_t(n, 3).abs().to(dev)
    k = n // 100
    t = torch.sort(sc, descending=True)[0][k - 1]
    spread = torch.randperm(n, generator=torch.Generator().manual_seed(ties))[:ties].to(dev)
    sc[spread] = t
    sc[n - 1] = t                                  # one of them in the last chunk
    above = int((sc > t).sum())
    n_eq = int((sc == t).sum())
    for need in (1, n_eq // 3, n_eq - 1, n_eq):
        mask = torch.full((n,), 7, dtype=torch.uint8, device=dev)
        res, _ = select_exact_device([sc], above + need, L.TIE_LOWEST_INDEX, masks=[mask])
        r = read_result(res)
        want, thresh, want_need, want_eq = _expected(sc, above + need)
        assert (r.status, r.n_selected, r.need, r.n_eq) == (0, above + need, want_need, want_eq)
        assert r.thresh == thresh and torch.equal(mask, want.to(torch.uint8)), need
