"""ptv3_voxelize where its parts, tiles and tables end, and ptv3_gather_rows over row widths."""
import numpy as np
import pytest
import torch

from gpu_util import DEV
from oracle import indexing as OI

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("sizes,grid,extent", [
    ([1], 0.02, 1.0), ([4095], 0.02, 1.0), ([4096], 0.02, 1.0), ([4097, 8191], 0.02, 1.0),   # edges of a tile
    ([3] * 1500, 0.02, 0.05),                     # many scenes inside a tile
    ([0, 5000, 0, 0, 3000, 0], 0.02, 1.0),
    ([131_072], 0.02, 3.0), ([131_073], 0.02, 3.0),   # 64 | 128 parts
    ([150_000, 100_000], 0.5, 1.0),               # a few voxels with thousands of points each: parts far over their table
    ([40_000], 10.0, 1.0),                        # one voxel
])
def test_voxelize_edges(sizes, grid, extent):
    from pointtransformerv3_amd import ops
    rng = np.random.default_rng(len(sizes) + sum(sizes))
    coord = np.concatenate([rng.random((n, 3)) * extent + rng.normal(0, 5, 3) for n in sizes]).astype(np.float32)
    offset = np.cumsum(sizes).astype(np.int64)
    wg, wi, winv, wends = OI.voxelize(coord, offset, grid)
    got = ops.voxelize(torch.from_numpy(coord).to(DEV), torch.from_numpy(offset).to(DEV), grid)
    for name, want in (("grid_coord", wg), ("index", wi), ("inverse", winv), ("offset", wends)):
        assert np.array_equal(got[name].cpu().numpy(), want), name


@pytest.mark.parametrize("n", [16 * 4096, 16 * 4096 + 1, 64 * 4096, 64 * 4096 + 1, 128 * 4096, 128 * 4096 + 1, 512 * 4096, 512 * 4096 + 1])
def test_voxelize_where_the_scan_down_the_tiles_takes_another_turn(n):
    """A thread of the scan has one tile | two of 16 shares; eight of 16 | three of 64 shares; eight of 64 in one trip | nine in two."""
    test_voxelize_edges([n - 5000, 5000], 0.05, 2.0)


@pytest.mark.parametrize("seed", [0, 9])
def test_voxelize_more_voxels_than_the_parts_tables_hold(seed):
    """14M voxels over 4096 parts: tables in memory. Against a sort of the voxel keys."""
    from pointtransformerv3_amd import ops
    n = 14_000_000
    gen = torch.Generator(device=DEV).manual_seed(3)
    g = torch.randint(0, 1200, (n, 3), generator=gen, device=DEV)
    g[0] = 0
    coord = (g.float() + 0.5)
    coord[0] = 0.0
    got = ops.voxelize(coord, torch.tensor([n], device=DEV), 1.0, seed=seed)
    key = (g[:, 0] * 1200 + g[:, 1]) * 1200 + g[:, 2]
    _, voxel, members = torch.unique(key, return_inverse=True, return_counts=True)
    idx, inv = got["index"], got["inverse"]
    assert len(idx) == len(members) and bool((idx[1:] > idx[:-1]).all())
    assert torch.equal(got["grid_coord"].long(), g[idx])
    assert torch.equal(key[idx[inv]], key)
    if seed == 0:
        first = torch.full_like(members, n).scatter_reduce(0, voxel, torch.arange(n, device=DEV), "amin")
        assert torch.equal(first.sort()[0], idx)


def test_gather_rows():
    from pointtransformerv3_amd import ops
    gen = torch.Generator().manual_seed(1)
    n = 3000
    for m in (1, 255, 256, 257, 2999):
        index = torch.randperm(n, generator=gen)[:m].sort()[0].to(DEV)
        many = [torch.randint(0, 256, (n, w), generator=gen, dtype=torch.uint8).to(DEV) for w in (1, 2, 3, 12, 16, 48, 2049, 4095, 4096)]
        many += [torch.randn(n, 3, generator=gen).to(DEV), torch.randn(n, 6, generator=gen).half().to(DEV),
                 torch.arange(n).to(DEV), torch.randn(n, 2, 2, generator=gen).double().to(DEV), torch.rand(n, 8, generator=gen).to(DEV)[:, 1:5]]
        for t, got in zip(many, ops.gather_rows(many, index)):
            assert got.dtype == t.dtype and torch.equal(got, t[index])
