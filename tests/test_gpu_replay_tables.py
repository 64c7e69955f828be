"""The replay's segment tables: tensors that begin and end inside a slab, and the
hand-over of learning rates and bias corrections to a step."""
import pytest
import torch

from oracle import trace as OT
from tests.util import same_bits, student_t

pytestmark = pytest.mark.gpu


def _rows(sizes, groups=1):
    rows, off = [], 0
    for i, s in enumerate(sizes):
        rows.append({"a": off, "n": s, "b1": (0.9, 0.8)[i % 2], "b2": (0.95, 0.99, 0.999)[i % 3],
                     "eps": (1e-8, 1e-6)[i % 2], "wd": 0.1 * (i % 2), "group": i % groups})
        off += s
    return rows, off


def _state(n, dev=None):
    gen = torch.Generator().manual_seed(n)
    p, m, v = torch.randn(n, generator=gen) * 0.02, torch.randn(n, generator=gen) * 1e-3, \
        torch.rand(n, generator=gen) * 1e-6
    return (p, m, v) if dev is None else (p.to(dev), m.to(dev), v.to(dev))


# one tensor; boundaries at, before and behind the ends of quads, slabs and workgroups; more tensors
# than a wave has lanes; more than travel in a step's arguments
_SIZES = [[1], [255], [256, 1], [1, 2, 3, 250, 256, 511, 1, 1], [1023, 1025, 3], [7] * 65 + [4000],
          [3] * 384, [3] * 385 + [5000], [1] * 2048, [2] * 2049]


@pytest.mark.parametrize("groups", [1, 3, 17])
@pytest.mark.parametrize("optimizer,bf16", [("adamw", True), ("adams", False)])
@pytest.mark.parametrize("sizes", _SIZES, ids=lambda s: f"{len(s)}x{sum(s)}")
def test_dense_steps_bit_for_bit(dev, sizes, optimizer, bf16, groups):
    """One chain of correctly rounded operations per coordinate: the oracle's bits.  The
    reconstruction is a sum in double whose order differs (n terms: n * 2^-53 relative)."""
    from sga_amd.replay_dense import DenseReplay
    rows, n = _rows(sizes, groups)
    w, m, v = _state(n)
    gs = [student_t(n, 5 + t).to(torch.bfloat16 if bf16 else torch.float32) for t in range(3)]
    metas = [{"clip_grad": 1.0, "grad_norm": 1.5, "lr": [1e-4 * (1 + t + i) for i in range(groups)]}
             for t in range(3)]
    lab, _, _, recon, _ = OT.dense_replay(rows, w, m, v, gs, metas, 7, (), optimizer)
    rep = DenseReplay(rows, *(t.to(dev) for t in _state(n)), 7, optimizer)
    for t, (g, meta) in enumerate(zip(gs, metas)):
        rep.step(t, g.to(dev), meta)
        got, want = rep.recon_steps[t]["recon_grad_norm"], recon[t]["recon_grad_norm"]
        assert abs(got - want) <= (n + 4) * 2.0 ** -53 * want
    # the oracle's in-place steps work on copies of the state: follow it to the end once more
    from oracle import replay as OR
    for t, (g, meta) in enumerate(zip(gs, metas)):
        for e in rows:
            a, b = e["a"], e["a"] + e["n"]
            OR.opt_step_inplace(g[a:b].float(), m[a:b], v[a:b], w[a:b], torch.zeros(e["n"]), meta["lr"][e["group"]],
                                e["wd"], e["b1"], e["b2"], *OR.bc_pair(optimizer, 7 + t + 1, e["b1"], e["b2"]),
                                e["eps"], optimizer=optimizer)
    for got, want in ((rep.w, w), (rep.m, m), (rep.v, v), (rep.label, lab)):
        assert same_bits(got, want)


@pytest.mark.parametrize("rows,sets", [(1, 1), (2, 2), (64, 16), (300, 3), (384, 16), (384, 17), (385, 1), (700, 700),
                                       (2048, 16), (2048, 17), (2049, 16)])
def test_first_kernel_writes_the_tables(dev, rows, sets):
    """Every row gets what the launch of its own gave it, on either side of what travels
    in a step's arguments (2048 rows, 16 different triples)."""
    from sga_amd import _lib as L
    from sga_amd.replay_dense import DenseReplay
    from sga_amd.replay_group import Config, ReplayGroup
    from sga_amd.segments import SegmentTable
    entries, n = _rows([5] * rows)
    for i, e in enumerate(entries):
        e.update(b1=0.9, b2=0.95, lr=1e-4 * (1 + i % sets), group=i % sets)
    g = student_t(n, 1).to(dev)
    group = ReplayGroup(entries, *_state(n, dev), [torch.ones(n, dtype=torch.bool, device=dev)],
                        [Config("abs_g", 10.0, 2)], 3, 9)
    dense = DenseReplay(entries, *_state(n, dev), 3)
    lrs = [1e-4 * (1 + i) for i in range(sets)]
    for t in range(2):
        group.step(g, {"clip_grad": 1.0, "grad_norm": 1.5, "lr": lambda e: e["lr"]})
        dense.step(t, g, {"clip_grad": 1.0, "grad_norm": 1.5, "lr": lrs})
        want = SegmentTable(entries, dev, start="a", segs=True, rsegs=True)
        want.refresh([e["lr"] for e in entries], 3 + t + 1)
        for got, ref in ((group._seg_table.segs, want.segs), (group._seg_table.rsegs, want.rsegs),
                         (dense._seg_table.rsegs, want.rsegs)):
            assert torch.equal(got, ref)
    ref = torch.empty_like(group.qn2)                   # pass 1 alone, on the same state
    out = [torch.empty_like(t) for t in (group.coef_d, group.coef_f)]
    group._fill_cfgs([False], {})
    args = (L.ptr(g), L.dtype_code(g), n, 1.0, 1.0, group._cfg_host, 1, L.ptr(group.partials))
    L.call("sga_replay_pass1", *args, L.ptr(ref), *map(L.ptr, out), L.stream())
    a, b, c = ref.clone(), out[0].clone(), out[1].clone()
    L.call("sga_replay_begin", *args, L.ptr(ref), *map(L.ptr, out), *group._seg_table.args, L.stream())
    assert torch.equal(a, ref) and torch.equal(b, out[0]) and torch.equal(c, out[1])
