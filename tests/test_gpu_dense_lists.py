"""The device check for dense per-crystal edge lists against the torch expressions it stands for (kept for tensors
it does not take), with the row offsets and pair lists that follow from it."""
import pytest
import torch

from crystalformer_amd import ops
from crystalformer_amd.encoder import get_edge_index
from oracle import torch_path as tp

pytestmark = pytest.mark.gpu

# one atom; ids with gaps in front, between and at the end of the atoms; sizes around a work-group of 256
SIZES = [[1], [2, 1, 3], [0, 0, 5, 0, 1, 4], [255, 1], [256], [257, 2], [16] * 40, [1] * 300, [300, 0, 0, 77]]


def tensors(sizes, dev):
    s = torch.tensor(sizes)
    edges = get_edge_index(s, torch.device("cuda", 0)) if dev.type == "cuda" else None
    return torch.repeat_interleave(torch.arange(len(sizes)), s).to(dev), edges


@pytest.mark.parametrize("sizes", SIZES)
def test_dense_lists_are_recognised(dev, sizes):
    batch, edges = tensors(sizes, dev)
    got = ops.dense_block_layout(batch, edges)
    want = ops.dense_block_layout(batch.cpu(), edges.cpu())
    assert got.dtype == torch.int64 and got.tolist() == want.tolist()
    pairs = ops.cached_edge_pairs(batch, edges, len(sizes))
    assert torch.equal(pairs, ops.edge_pairs(got))
    N = batch.numel()
    assert torch.equal(ops.cached_edge_row_offsets(edges, N).cpu(), tp.edge_row_offsets(edges.cpu(), N))
    assert torch.equal(ops.cached_edge_row_offsets(edges, N), ops.edge_row_offsets(edges, N))
    atom_start, edge_start = ops.cached_crystal_offsets(batch)
    assert atom_start.tolist() == [0] + got.cumsum(0).tolist()
    assert edge_start.tolist() == [0] + (got * got).cumsum(0).tolist()


@pytest.mark.parametrize("sizes", [[2, 1, 3], [255, 1], [16] * 40])
def test_other_lists_are_not(dev, sizes):
    batch, edges = tensors(sizes, dev)
    E = edges.shape[1]
    wrong = []
    for row, at in ((0, 0), (1, 0), (0, E - 1), (1, E - 1), (1, E // 2)):
        other = edges.clone()
        other[row, at] = (other[row, at] + 1) % batch.numel()
        wrong.append((batch, other))
    wrong += [(batch, edges[:, :-1].contiguous()), (batch, torch.cat([edges, edges[:, -1:]], 1)),
              (batch, edges.flip(0).contiguous()), (batch, edges[:, :0].contiguous()), (batch.flip(0).contiguous(), edges),
              (batch - 1, edges), (batch + (1 << 24), edges), (torch.zeros_like(batch), edges)]
    for b, e in wrong:
        assert ops.dense_block_layout(b.cpu(), e.cpu()) is None
        assert ops.dense_block_layout(b, e) is None
        assert ops.cached_edge_pairs(b, e, 1 << 24) is None
    # (forms the device check leaves to torch)
    spread = torch.empty(2, 2 * E, dtype=torch.int64, device=dev)[:, ::2]
    spread.copy_(edges)
    assert ops.dense_block_layout(batch, spread).tolist() == sizes


# either side of the crystal counts up to which one work-group scans them
@pytest.mark.parametrize("crystals", [ops.SCAN_TWO, ops.SCAN_TWO + 1, ops.SCAN_THREE + 1, ops.SCAN_DENSE + 1])
def test_many_crystals(dev, crystals, monkeypatch):
    g = torch.Generator().manual_seed(crystals)
    sizes = torch.randint(0, 4, (crystals,), generator=g)
    sizes[-1] = 3
    batch = torch.repeat_interleave(torch.arange(crystals), sizes).to(dev)
    scans = []
    scan = ops._lib.load().cf_layout_scan
    monkeypatch.setattr(ops._lib.load(), "cf_layout_scan", lambda *a: scans.append(a[1]) or scan(*a))
    edges, _ = ops.edge_index(sizes.to(dev))
    assert len(scans) == (crystals <= ops.SCAN_TWO)
    pairs = ops.edge_pairs(sizes.to(dev))
    assert len(scans) == (crystals <= ops.SCAN_TWO) + (crystals <= ops.SCAN_THREE)
    N = batch.numel()
    start = torch.cat([torch.zeros(1, dtype=torch.int64), sizes.cumsum(0)])[batch.cpu()]
    rows = torch.repeat_interleave(torch.arange(N), sizes[batch.cpu()])
    first = torch.cat([torch.zeros(1, dtype=torch.int64), sizes[batch.cpu()].cumsum(0)])[:-1]
    assert torch.equal(edges[0].cpu(), rows)
    assert torch.equal(edges[1].cpu(), start[rows] + torch.arange(rows.numel()) - first[rows])
    assert ops.dense_block_layout(batch, edges).tolist() == sizes.tolist()
    assert torch.equal(ops.cached_edge_pairs(batch, edges, crystals), pairs)
    edges[1, 5] += 1
    assert ops.dense_block_layout(batch, edges) is None
