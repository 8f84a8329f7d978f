"""Tile emission and the stable sort at the edges of a wave's run and of the
radix tiles, against a plain enumeration."""

import pytest
import torch

from r2splat_amd import hip as ops

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("dtype", [torch.float32, torch.float64])
@pytest.mark.parametrize("n,largest,tiles", [(1, 9, (3, 4, 5)), (63, 1, (3, 4, 5)), (64, 40, (5, 1, 7)), (65, 2, (1, 1, 1)),
                                             (1000, 3, (16, 17, 18)), (4000, 30, (9, 8, 7)), (20_000, 9, (16, 16, 16))])
def test_isect_tiles_3d_lists_every_box_in_order(device, n, largest, tiles, dtype):
    nx, ny, nz = tiles
    g = torch.Generator().manual_seed(n)
    size = torch.tensor([8.0 * nx, 8.0 * ny, 8.0 * nz], dtype=torch.float64)
    means = ((torch.rand(n, 3, generator=g, dtype=torch.float64) * 1.4 - 0.2) * size).to(dtype)
    # a third of the primitives reach no tile (a zero radius), some lie outside
    radii = torch.randint(1, largest + 1, (n, 3), generator=g, dtype=torch.int32)
    radii[torch.rand(n, generator=g) < 0.33, 1] = 0
    counts, ids, flat = ops.isect_tiles_3d(means.to(device), radii.to(device), 8, nx, ny, nz)
    m, r = means / 8, radii.to(dtype) / 8
    limit = torch.tensor([nx, ny, nz], dtype=dtype)
    lo = torch.minimum(torch.floor(m - r).clamp(min=0), limit).long()
    hi = torch.minimum(torch.ceil(m + r).clamp(min=0), limit).long()
    lo[(radii <= 0).any(1)] = 0
    hi[(radii <= 0).any(1)] = 0
    span = (hi - lo).clamp(min=0)
    number = span.prod(1)
    assert torch.equal(counts.cpu().long(), number)
    owner = torch.repeat_interleave(torch.arange(n), number)
    k = torch.arange(len(owner)) - torch.repeat_interleave(torch.cumsum(number, 0) - number, number)
    w, wh = span[owner, 0], span[owner, 0] * span[owner, 1]
    x, y, z = k % w, k % wh // w, k // wh
    key = ((lo[owner, 2] + z) * ny + lo[owner, 1] + y) * nx + lo[owner, 0] + x
    key, order = torch.sort(key, stable=True)
    assert torch.equal(ids.cpu(), key)
    assert torch.equal(flat.cpu().long(), owner[order])
