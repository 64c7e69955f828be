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
