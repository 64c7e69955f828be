"""What a caller changes between steps -- learning rates, hyper-parameters, pack
buffers -- and what of it the next step has to see."""
import pytest
import torch

pytestmark = pytest.mark.gpu

N = 5000


def _rows(key):
    return [{key: 0, "n": 2000, "lr": 1e-3, "b1": 0.9, "b2": 0.95, "eps": 1e-8, "wd": 0.1, "group": 0},
            {key: 2000, "n": 3000, "lr": 1e-3, "b1": 0.9, "b2": 0.95, "eps": 1e-8, "wd": 0.0, "group": 0}]


def _table(t, row_type, count=2):
    return (row_type * count).from_buffer_copy(bytes(t.cpu().numpy()))


def _flat(dev, seed, scale):
    return torch.randn(N, generator=torch.Generator().manual_seed(seed)).mul_(scale).to(dev)


def _state(dev):
    return _flat(dev, 1, 0.02), _flat(dev, 2, 1e-3), _flat(dev, 3, 1e-3).square_()


def _stepper(dev, rows, **kw):
    from sga_amd.fused_step import FusedSparseStep
    fs = FusedSparseStep(N, rows, dev, max_k=N, **kw)
    state = [torch.zeros(N, device=dev), *_state(dev)]
    return fs, lambda step: fs.step(_flat(dev, 10 + step, 1e-2), *state, step, k=50)


def test_a_list_of_learning_rates_changed_in_place(dev):
    from sga_amd import _lib as L
    from sga_amd.segments import SegmentTable
    table = SegmentTable(_rows("start"), dev)
    lr = [1e-3, 2e-3]
    table.refresh(lr, 1)
    lr[1] = 5e-4
    table.refresh(lr, 2)
    assert [r.lr for r in _table(table.segs, L.Segment)] == [L.f32(1e-3), L.f32(5e-4)]


@pytest.mark.parametrize("kind", ["group", "dense"])
def test_replay_follows_its_entries(dev, kind):
    from sga_amd import _lib as L
    from sga_amd.replay_dense import DenseReplay
    from sga_amd.replay_group import Config, ReplayGroup
    from sga_amd.segments import ReplaySegment
    rows, (w, m, v) = _rows("a"), _state(dev)
    meta = {"clip_grad": 1.0, "grad_norm": float("nan"), "lr": 1e-4 if kind == "group" else [1e-4]}
    if kind == "group":
        rep = ReplayGroup(rows, w, m, v, [torch.ones(N, dtype=torch.uint8, device=dev)],
                          [Config("abs_g", 10.0, 4)], 3, 4)
        step = lambda i: rep.step(_flat(dev, i, 1e-2), meta)                  # noqa: E731
    else:
        rep = DenseReplay(rows, w, m, v, 3)
        step = lambda i: rep.step(i, _flat(dev, i, 1e-2), meta)               # noqa: E731
    step(0)
    rows[0].update(wd=0.3, eps=1e-6)
    rows[1].update(b1=0.8, b2=0.99)
    step(1)
    for t, row_type in ((rep._seg_table.rsegs, ReplaySegment), (rep._seg_table.segs, L.Segment)):
        if t is None:
            continue
        for got, r in zip(_table(t, row_type), rows):
            assert (got.start, got.n) == (r["a"], r["n"])
            want = (r["b1"], 1 - r["b1"], r["b2"], 1 - r["b2"], r["eps"], 1 - r["b1"] ** 5, 1 - r["b2"] ** 5)
            assert (got.beta1, got.om1, got.beta2, got.om2, got.eps, got.bc1, got.bc2) == \
                tuple(L.f32(x) for x in want)
            assert got.wd == (r["wd"] if row_type is ReplaySegment else L.f32(r["wd"]))
            assert row_type is L.Segment or got.wdf == L.f32(r["wd"])


def test_fused_step_takes_the_bias_corrections_of_its_segments(dev):
    """Learning rates and bias corrections follow the segments; betas, eps and weight
    decay are those the stepper was made with."""
    from sga_amd import _lib as L
    rows = _rows("start")
    fs, step = _stepper(dev, rows)
    step(1)
    rows[1].update(lr=5e-4, b1=0.8, b2=0.99, wd=0.7)
    step(2)
    got = _table(fs._seg_dev, L.Segment)[1]
    assert (got.lr, got.bc1, got.bc2) == (L.f32(5e-4), L.f32(1 - 0.8 ** 2), L.f32(1 - 0.99 ** 2))
    assert (got.beta1, got.beta2, got.wd) == (L.f32(0.9), L.f32(0.95), 0.0)


def test_the_returned_pack_is_of_the_present_buffers(dev):
    fs, step = _stepper(dev, _rows("start"))
    idx, val = step(1)
    idx.resize_(10)                                     # the caller's own view, done with as it likes
    assert step(2)[0].shape == (50,)
    fs.idx, fs.values = torch.empty_like(fs.idx), torch.empty_like(fs.values)
    idx, val = step(3)
    assert (idx.data_ptr(), val.data_ptr()) == (fs.idx.data_ptr(), fs.values.data_ptr())
    assert idx.shape == val.shape == (50,) and bool((idx[1:] > idx[:-1]).all())
