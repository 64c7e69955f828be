"""The table-driven launches of the plugin steps (clip norm, clip scale, commits)
against the per-tensor entry points and float64, at the edges of their
4096-element spans and of the 64-record rounds of the table search."""
from types import SimpleNamespace

import pytest
import torch

pytestmark = pytest.mark.gpu

EDGES = [1, 3, 4095, 4096, 4097, 8192, 12_289]


def _records(dev, sizes, seed, with_mask):
    from sga_amd.adamw import ParamRecord
    gen = torch.Generator().manual_seed(seed)
    n = sum(sizes)
    t = {k: (torch.randn(n, generator=gen) * s).to(dev) for k, s in
         (("p", 0.02), ("g", 1e-2), ("m", 1e-3))}
    t["v"] = (torch.rand(n, generator=gen) * 1e-4).to(dev)
    mask = (torch.rand(n, generator=gen) < 0.03).to(torch.uint8).to(dev) if with_mask else None
    bucket = SimpleNamespace(active_mask_u8=mask, grad_data=t["g"], extra_main_grads=[], support_index=0)
    recs, off = [], 0
    for i, s in enumerate(sizes):
        e = slice(off, off + s)
        recs.append(ParamRecord(None, SimpleNamespace(data=t["p"][e], grad=t["g"][e]), bucket, off, off + s,
                                1e-3, 0.9, 0.95, 1e-8, 0.1 * (i % 2), 7,
                                _state={"exp_avg": t["m"][e], "exp_avg_sq": t["v"][e]}))
        off += s
    return recs, t, mask


# 63 / 64 / 65 records: one and two rounds of the search; odd sizes shift every later record off
# 16-byte alignment and leave remainders, which go element by element
@pytest.mark.parametrize("count", [1, 7, 63, 64, 65, 200])
@pytest.mark.parametrize("with_mask", [True, False])
def test_clip_tables(dev, count, with_mask):
    from sga_amd.clip import masked_clip_grad_norm
    sizes = [EDGES[i % len(EDGES)] for i in range(count)]
    recs, t, mask = _records(dev, sizes, count, with_mask)
    before = t["g"].clone()
    on = before if mask is None else before * mask
    exact = float(on.double().square().sum().sqrt())
    norm, coeff = masked_clip_grad_norm(recs, 0.5 * exact, was_full=False, trace_dumps=with_mask)
    # fp32 partials of 4096 squares each, folded in double: below 4096 * 2^-24 relative
    assert abs(norm - exact) <= 2.5e-4 * exact
    if with_mask:                                # dump steps scale in place
        c32 = torch.tensor(0.5 * exact / (norm + 1e-6), device=dev)
        assert coeff == 1.0 and torch.equal(t["g"], torch.where(mask > 0, before * c32, before))


# the last element of every record carries the norm: a remainder that was left out would show
@pytest.mark.parametrize("count", [1, 7, 63, 64, 65, 200])
@pytest.mark.parametrize("was_full", [True, False])
def test_clip_reaches_every_record_end(dev, count, was_full):
    from sga_amd import _lib as L
    from sga_amd.clip import masked_clip_grad_norm
    sizes = [EDGES[i % len(EDGES)] for i in range(count)]
    recs, t, mask = _records(dev, sizes, 300 + count, not was_full)
    ends = torch.tensor(sizes).cumsum(0).to(dev) - 1
    t["g"][ends] = 10.0 + torch.arange(count, device=dev) % 3
    if mask is not None:
        mask[ends] = 1
    before = t["g"].clone()
    exact = float((before if mask is None else before * mask).double().square().sum().sqrt())
    assert len(L.host().norm_table(recs, was_full)) == 4          # the launches over the table, no other route
    norm, coeff = masked_clip_grad_norm(recs, 0.5 * exact, was_full=was_full, trace_dumps=not was_full)
    # a square is rounded, then added at most 16 + 6 + 2 times in fp32 (lane, wave, workgroup), then in double;
    # the sum, its root and the result are rounded once each
    assert abs(norm - exact) <= (25 / 2 + 2) * 2.0 ** -24 * exact
    c32 = torch.tensor(0.5 * exact / (norm + 1e-6), device=dev)
    want = before * c32 if mask is None else torch.where(mask > 0, before * c32, before)
    assert coeff == 1.0 and torch.equal(t["g"], want)


@pytest.mark.parametrize("count", [1, 7, 64, 65, 200])
@pytest.mark.parametrize("phase", ["full", "sparse", "sparse_fold", "compact"])
def test_commit_tables(dev, count, phase):
    from sga_amd import config
    from sga_amd.adamw import (OptContext, SgaAdamW, adamw_grad_correct, adamw_grad_correct_compact,
                               build_dir_table)
    from sga_amd.support import compact_mask_u8
    config.set_args(SimpleNamespace(sga_score="update", sga_optimizer_residual_mean=True,
                                    sga_optimizer_compact_search="table",
                                    sga_optimizer_full_sync_inactive_lr_scale=1.0))
    sizes = [EDGES[i % len(EDGES)] for i in range(count)]
    recs, t, mask = _records(dev, sizes, 100 + count, phase != "full")
    ref_recs, ref, _ = _records(dev, sizes, 100 + count, phase != "full")
    opt, kw = SgaAdamW(), {}
    if phase == "compact":
        idx = compact_mask_u8(mask)
        vals = t["g"][idx.long()].contiguous()
        table = build_dir_table(idx, sum(sizes))
        kw = dict(compact_values={id(recs[0].bucket_state): vals},
                  support=SimpleNamespace(buckets=[SimpleNamespace(idx=idx, dir_table=table)]))
    ctx = OptContext(recs, phase, bucket_states=[recs[0].bucket_state], apply_coeff=0.5, fold_window=4,
                     next_step_is_full=phase == "sparse_fold", **kw)
    (opt.full_step if phase == "full" else opt.sparse_step)(ctx)
    for r in ref_recs:
        a = (r.main_param.data, r.grad, r.m, r.v)
        h = (r.lr, r.beta1, r.beta2, r.eps, r.weight_decay, r.step)
        if phase == "full":
            adamw_grad_correct(*a, *h, emit_score="update")
        elif phase == "compact":
            adamw_grad_correct_compact(*a, idx, vals, r.start, *h, coeff=0.5, dir_table=table)
        else:
            adamw_grad_correct(*a, *h, mask=r.mask_u8(), coeff=0.5, clear=True,
                               fold=phase == "sparse_fold", interval=4.0)
    for k in t:
        assert torch.equal(t[k], ref[k]), k


@pytest.mark.parametrize("phase", ["sparse", "compact"])
def test_a_captured_commit_keeps_its_table(dev, phase):
    """Replays read the staged table again: nothing that the program stages between them may get there."""
    from sga_amd import config
    from sga_amd import adamw as A
    from sga_amd.support import compact_mask_u8
    config.set_args(SimpleNamespace(sga_score="update", sga_optimizer_residual_mean=False,
                                    sga_optimizer_compact_search="table",
                                    sga_optimizer_full_sync_inactive_lr_scale=1.0))
    sizes = [4097, 12_289, 3]
    recs, t, mask = _records(dev, sizes, 9, True)
    refs, ref, _ = _records(dev, sizes, 9, True)
    kw = {}
    if phase == "compact":
        idx = compact_mask_u8(mask)
        vals = t["g"][idx.long()].contiguous()
        table = A.build_dir_table(idx, sum(sizes))
        kw = dict(support=SimpleNamespace(buckets=[SimpleNamespace(idx=idx, dir_table=table)]))
    opt = A.SgaAdamW()

    def step(rs):
        if kw:
            kw["compact_values"] = {id(rs[0].bucket_state): vals}
        opt.sparse_step(A.OptContext(rs, "sparse", bucket_states=[rs[0].bucket_state], apply_coeff=0.5, **kw))
    warm, _, _ = _records(dev, sizes, 10, True)         # the general route lays its staging out once
    walk, A.L.capturing = A.L.capturing, lambda: True
    try:
        step(warm)
    finally:
        A.L.capturing = walk
    torch.cuda.synchronize()
    graph = torch.cuda.CUDAGraph()
    with torch.cuda.graph(graph):
        step(recs)
    for turn in range(3):
        staged = [torch.full((1 << b,), 0, dtype=torch.uint8, pin_memory=True) for b in range(7, 14)]
        graph.replay()
        torch.cuda.synchronize()
        step(refs)
        for k in t:
            assert torch.equal(t[k], ref[k]), (k, turn)
        del staged


@pytest.mark.parametrize("entries", [0, 1])
def test_a_directory_table_too_short_is_refused(dev, entries):
    from sga_amd import config
    from sga_amd.adamw import OptContext, SgaAdamW
    from sga_amd.support import compact_mask_u8
    config.set_args(SimpleNamespace(sga_score="update", sga_optimizer_residual_mean=False,
                                    sga_optimizer_compact_search="table",
                                    sga_optimizer_full_sync_inactive_lr_scale=1.0))
    recs, t, mask = _records(dev, [4097], 3, True)
    idx = compact_mask_u8(mask)
    bucket = SimpleNamespace(idx=idx, dir_table=torch.zeros(entries, dtype=torch.int32, device=dev))
    ctx = OptContext(recs, "sparse", bucket_states=[recs[0].bucket_state],
                     compact_values={id(recs[0].bucket_state): t["g"][idx.long()].contiguous()},
                     support=SimpleNamespace(buckets=[bucket]))
    before = t["p"].clone()
    with pytest.raises(AssertionError, match="dir_table"):
        SgaAdamW().sparse_step(ctx)
    assert torch.equal(t["p"], before)


# a launch writes 64 or 240 rows: one short of, at and past both, and several launches
@pytest.mark.parametrize("count", [1, 63, 64, 65, 239, 240, 241, 500])
def test_segment_table_refresh(dev, count):
    import ctypes
    from sga_amd import _lib as L
    from sga_amd.segments import ReplaySegment, SegmentTable
    rows = [dict(start=17 * i, n=17, b1=(0.9, 0.8)[i % 2], b2=0.95 + 0.01 * (i % 3), eps=1e-8, wd=0.1 * (i % 2))
            for i in range(count)]
    table = SegmentTable(rows, dev, segs=True, rsegs=True)
    for step, lr in ((1, 1e-4), (7, [1e-3 * (1 + i) for i in range(count)]), (8, 2e-4)):
        table.refresh(lr, step)
        got = (L.Segment * count).from_buffer_copy(bytes(table.segs.cpu().numpy()))
        rgot = (ReplaySegment * count).from_buffer_copy(bytes(table.rsegs.cpu().numpy()))
        for i, r in enumerate(rows):
            x = lr if isinstance(lr, float) else lr[i]
            want = [r["start"], r["n"]] + [L.f32(v) for v in (
                x, r["b1"], 1.0 - r["b1"], r["b2"], 1.0 - r["b2"], r["eps"], r["wd"], 1.0 - r["b1"] ** step,
                1.0 - r["b2"] ** step)]
            assert [getattr(got[i], f[0]) for f in got[i]._fields_][:-1] == want, (step, i)
            assert (rgot[i].lr, rgot[i].wd, rgot[i].bc1, rgot[i].bc2, rgot[i].om2) == \
                (x, r["wd"], want[-2], want[-1], want[6]), (step, i)
    assert ctypes.sizeof(L.Segment) * count == table.segs.numel()
