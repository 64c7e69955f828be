"""The score that a full commit leaves for the select, on both sides of the
size up to which it stays in the memory-side cache, at odd starts and lengths."""
from types import SimpleNamespace

import pytest
import torch

from tests.util import same_bits

pytestmark = pytest.mark.gpu
LINE = (288 << 20) // 4


def _records(n, dev, first, gen):
    from sga_amd.adamw import ParamRecord
    p, g, m, v = (torch.randn(n, generator=gen, device=dev) * s for s in (0.02, 1e-3, 1e-4, 1e-6))
    v.abs_()
    recs = []
    for a, b in ((0, first), (first, n)):
        mp = SimpleNamespace(data=p[a:b], grad=g[a:b])
        recs.append(ParamRecord(None, mp, SimpleNamespace(active_mask_u8=None), a, b, 1e-3, 0.9, 0.95, 1e-8, 0.1, 3,
                                _state={"exp_avg": m[a:b], "exp_avg_sq": v[a:b]}))
    return recs, (p, g, m, v)


@pytest.mark.parametrize("score", ["abs_g", "update", "coi", "abs_m"])
@pytest.mark.parametrize("n,first", [(4096, 1), (70_001, 4096), (1_000_003, 12_345)])
def test_every_score_is_whole(dev, n, first, score):
    """Against the same commit a record at a time (its own kernel)."""
    from sga_amd import _lib as L
    from sga_amd.adamw import SCORE_MAP, OptContext, SgaAdamW
    from sga_amd.config import set_args
    set_args(SimpleNamespace(sga_score=score, sga_optimizer_residual_mean=False, sga_optimizer_compact_search="table",
                             sga_optimizer_full_sync_inactive_lr_scale=1.0))
    ends = []
    for multi in (True, False):
        gen = torch.Generator(device=dev).manual_seed(n)
        recs, state = _records(n, dev, first, gen)
        if multi:
            SgaAdamW().full_step(OptContext(recs, "full", bucket_states=[]))
        else:
            emit = SCORE_MAP[score]
            p, g, m, v = state
            for r in recs:
                a, b = r.start, r.end
                L.call("sga_adamw_grad_correct", L.ptr(p[a:b]), L.ptr(g[a:b]), L.ptr(m[a:b]), L.ptr(v[a:b]), None, b - a,
                       1e-3, 0.9, 1.0 - 0.9, 0.95, 1.0 - 0.95, 1e-8, 0.1, 1.0 - 0.9 ** 3, 1.0 - 0.95 ** 3, 1.0, 1.0,
                       1e-3, emit, 0, L.stream())
        ends.append(state)
    for a, b in zip(*ends):
        assert same_bits(a, b)


@pytest.mark.parametrize("n", [LINE - 4096, LINE, LINE + 4096])
def test_scores_around_the_line(dev, n):
    """|g| and |m| are bits of the inputs."""
    from sga_amd.adamw import OptContext, SgaAdamW
    from sga_amd.config import set_args
    for score, which in (("abs_g", 1), ("abs_m", 2)):
        set_args(SimpleNamespace(sga_score=score, sga_optimizer_residual_mean=False, sga_optimizer_compact_search="table",
                                 sga_optimizer_full_sync_inactive_lr_scale=1.0))
        recs, state = _records(n, dev, 4096 * 1000, torch.Generator(device=dev).manual_seed(n))
        want = state[which].abs()
        SgaAdamW().full_step(OptContext(recs, "full", bucket_states=[]))
        assert torch.equal(state[1], want)
        del recs, state, want
