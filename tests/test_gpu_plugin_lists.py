"""Pack and unpack of the plugin layouts in one launch each: slice bounds with the pack, values with the
positions, slices from arrays of their own."""
import pytest
import torch

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("k", [1, 2, 63, 64, 65, 4096, 4097, 70_000])
@pytest.mark.parametrize("where", ["low", "high", "both"])
def test_bounds_come_with_the_pack(dev, k, where):
    from sga_amd.backends import index_layout_bounds, index_layout_pack
    n = 4 * k + 3
    gen = torch.Generator().manual_seed(k)
    lo, hi = {"low": (0, n // 2), "high": (n // 2, n), "both": (0, n)}[where]
    idx = (torch.randperm(hi - lo, generator=gen)[:k] + lo).sort().values.to(torch.int32).to(dev)
    grad = torch.randn(n, generator=gen).to(dev)
    for slices in (2, 3):
        g, values = grad.clone(), torch.full((idx.numel(),), -1.0, device=dev)
        out = index_layout_pack(g, idx, values, factor=0.5, slices=slices)
        assert out == index_layout_bounds(idx, n, slices)
        assert torch.equal(values, grad[idx.long()] * 0.5)
        want = grad.clone()
        want[idx.long()] = 0
        assert torch.equal(g, want)


def _mask(n, density, gen):
    if density == "ends":
        m = torch.zeros(n, dtype=torch.uint8)
        m[0] = m[-1] = 1
        return m
    return (torch.rand(n, generator=gen) < density).to(torch.uint8) * 3      # any non-zero byte counts


# one and several chunks, groups of 16 chunks, and rounds of 1024 groups, whole and ragged
@pytest.mark.parametrize("n", [1, 17, 1024, 16 * 1024 - 1, 16 * 1024 + 1, 1_150_187, 1024 * 16 * 1024 + 5])
@pytest.mark.parametrize("density", [0.0, "ends", 0.01, 0.3, 1.0])
def test_mask_lists(dev, n, density):
    from sga_amd.backends import mask_layout_pack, mask_layout_unpack
    from sga_amd.support import compact_mask_u8
    gen = torch.Generator().manual_seed(n % 1000)
    mask = _mask(n, density, gen).to(dev)
    grad = torch.randn(n, generator=gen).to(dev)
    at = mask.nonzero().reshape(-1)
    assert torch.equal(compact_mask_u8(mask), at.to(torch.int32))
    for slices in (2, 3, 8, 9):
        payloads, idx = mask_layout_pack(grad, mask, factor=0.5, slices=slices)
        cuts = [i * (n // slices) for i in range(slices)] + [n]
        assert torch.equal(idx, at.to(torch.int32)) and len(payloads) == slices
        for p, a, b in zip(payloads, cuts[:-1], cuts[1:]):
            assert torch.equal(p, grad[a:b][mask[a:b] != 0] * 0.5)
        dst = torch.zeros(n, device=dev)
        mask_layout_unpack(dst, idx, payloads)
        assert torch.equal(dst, torch.where(mask != 0, grad * 0.5, torch.zeros_like(grad)))


def test_mask_lists_on_views(dev):
    from sga_amd.backends import mask_layout_pack
    gen = torch.Generator().manual_seed(3)
    grad, mask = torch.randn(70_003, generator=gen).to(dev), _mask(70_003, 0.1, gen).to(dev)
    for off in (1, 2, 3, 5):
        payloads, idx = mask_layout_pack(grad[off:], mask[off:], slices=2)
        assert torch.equal(torch.cat(payloads), grad[off:][mask[off:] != 0])
        assert torch.equal(idx.long(), mask[off:].nonzero().reshape(-1))


@pytest.mark.parametrize("slices", [0, -1])
def test_no_slices_pack_nothing(dev, slices):
    from sga_amd.backends import index_layout_pack
    grad, values = torch.ones(9, device=dev), torch.zeros(5, device=dev)
    assert index_layout_pack(grad, torch.arange(5, dtype=torch.int32, device=dev), values, slices=slices) == []
    assert grad.sum().item() == 9 and values.sum().item() == 0


@pytest.mark.parametrize("k", [(8 << 20) - 1, 8 << 20, (8 << 20) + 1])
def test_long_lists_in_parts(dev, k):
    """Around the number of entries from which the parts are launches of their own."""
    from sga_amd.kernels import scatter_parts
    gen = torch.Generator(device=dev).manual_seed(k)
    idx = torch.arange(k, dtype=torch.int32, device=dev) * 2
    values = torch.randn(k, generator=gen, device=dev)
    dst = torch.zeros(2 * k, device=dev)
    scatter_parts(dst, idx, [values[:5].clone(), values[5:k // 2 + 3].clone(), values[k // 2 + 3:].clone()])
    assert torch.equal(dst[::2], values) and not bool(dst[1::2].any())


# rounds of the workgroup that adds up: of 1024 groups of 16 K bytes a thread each, of 16 K by runs of sixteen
@pytest.mark.parametrize("n", [2 ** 24, 2 ** 24 + 1, 1040 * 2 ** 14 - 3, 1041 * 2 ** 14, 2 ** 28, 2 ** 28 + 1,
                               3 * 2 ** 28 + 123_457])
def test_long_masks(dev, n):
    from sga_amd.support import compact_mask_u8
    mask = torch.zeros(n, dtype=torch.uint8, device=dev)
    on = torch.cat([torch.randint(0, n, (50_000,), generator=torch.Generator().manual_seed(n % 1009)),
                    torch.arange(n - 40_000, n), torch.arange(0, n, 2 ** 14)]).unique().to(dev)
    mask[on] = 2
    idx, before = compact_mask_u8(mask, step=n // 3, cuts=3)
    assert torch.equal(idx, on.to(torch.int32))
    assert before == [int((on < (j + 1) * (n // 3)).sum()) for j in range(3)]
