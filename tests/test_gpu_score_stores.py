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


@pytest.mark.parametrize("n,configs", [(5_000_000, 2), (15 << 20, 1), ((15 << 20) + 1, 1)])
def test_replay_steps_around_their_line(dev, n, configs):
    """Steps of several configurations against each of them alone (fewer bytes a step), dense steps against
    the commit in torch."""
    from sga_amd.replay_dense import DenseReplay
    from sga_amd.replay_group import Config, ReplayGroup
    gen = torch.Generator(device=dev).manual_seed(n)
    w, m = (torch.randn(n, generator=gen, device=dev) * s for s in (0.02, 1e-4))
    v = torch.rand(n, generator=gen, device=dev) * 1e-6 + 1e-8
    entries = [{"a": 0, "n": n - 1000, "b1": 0.9, "b2": 0.95, "eps": 1e-8, "wd": 0.1, "group": 0},
               {"a": n - 1000, "n": 1000, "b1": 0.8, "b2": 0.99, "eps": 1e-6, "wd": 0.0, "group": 0}]
    steps = [(torch.randn(n, generator=gen, device=dev) * 1e-3).to(torch.bfloat16) for _ in range(3)]
    meta = {"clip_grad": 1.0, "grad_norm": 1.5, "lr": 1e-4}
    arms = [Config("abs_g", 1.0, 2), Config("abs_g_blind", 2.0, 4)][:configs]
    sel = [torch.rand(n, generator=gen, device=dev) < 0.01 for _ in arms]

    def run(which):
        group = ReplayGroup(entries, w, m, v, [sel[j] for j in which], [arms[j] for j in which], t0=5, window=1 << 10)
        for g in steps:
            group.step(g, meta)
        return [(st.data.clone(), st.sel.clone()) for st in group.state]
    together = run(range(configs))
    for j in range(configs):
        (data, picked), = run([j])
        assert same_bits(together[j][0], data) and torch.equal(together[j][1], picked)
    dense = DenseReplay(entries, w, m, v, 5, "adamw")
    for t, g in enumerate(steps):
        dense.step(t, g, dict(meta, lr=[1e-4]))
    pm, pv = m.clone(), v.clone()
    for g in steps:
        q = g.float()
        pm[:n - 1000] = pm[:n - 1000] * 0.9 + q[:n - 1000] * 0.1
        pv[:n - 1000] = pv[:n - 1000] * 0.95 + q[:n - 1000] ** 2 * 0.05
    # three roundings a step of each moment
    assert torch.allclose(dense.m[:n - 1000], pm[:n - 1000], rtol=1e-6, atol=1e-10)
    assert torch.allclose(dense.v[:n - 1000], pv[:n - 1000], rtol=1e-6, atol=1e-16)
