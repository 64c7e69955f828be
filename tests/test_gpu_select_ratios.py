"""Selects at ratios where the sampled bracket ends at the edges of histogram bins, at the edges of their
parts, and at keys; lists with one to dozens of entries a chunk."""
import pytest
import torch

from tests.util import student_t

pytestmark = pytest.mark.gpu


def _scores(kind, n):
    sc = student_t(n, n % 89).abs()
    if kind == "bf16":
        return sc.to(torch.bfloat16).float()
    if kind == "runs":                     # the largest lie side by side: chunks full of list entries beside empty ones
        head = sc[:n // 8].sort(descending=True).values
        return torch.cat([sc[n // 8:], head])
    return sc


@pytest.mark.parametrize("kind", ["student", "bf16", "runs"])
@pytest.mark.parametrize("n", [1025, 150_001, 1_000_003, 8192 * 1024, 8192 * 1024 + 3])
def test_selects_by_ratio(dev, n, kind):
    from sga_amd import _lib as L
    from sga_amd.selection import read_result, select_exact_device
    sc = _scores(kind, n).to(dev)
    order = torch.sort(sc, descending=True).values
    for ratio in (0.01, 0.3, 1.0, 7.0, 10.0, 13.0, 40.0):
        k = max(1, int(n * ratio / 100))
        t = order[k - 1]
        want = sc > t
        need = k - int(want.sum())
        want[(sc == t).nonzero().reshape(-1)[:need]] = True
        mask = torch.full((n,), 7, dtype=torch.uint8, device=dev)
        res, _ = select_exact_device([sc], k, L.TIE_LOWEST_INDEX, masks=[mask])
        r = read_result(res)
        assert (r.status, r.n_selected, r.need, r.thresh) == (0, k, need, float(t)), (ratio, vars(r))
        assert torch.equal(mask, want.to(torch.uint8)), ratio
