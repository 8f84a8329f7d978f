"""The fused prepare at the edges of its rules: the primitive order on both
sides of its one-workgroup size and of its radix tiles, and the binning with
short and long ranges, small and large bin tables and the sort, against the
float64 operator binning."""

import pytest
import torch

from r2splat_amd import fused, hip as ops, workloads

pytestmark = pytest.mark.gpu


def _codes(means, n):
    lo, hi = means.min(0).values, means.max(0).values
    q = torch.nan_to_num((means - lo) / (hi - lo) * 32).clamp(0, 31).long()
    code = torch.zeros(n, dtype=torch.long, device=means.device)
    for bit in range(5):
        for k in range(3):
            code |= ((q[:, k] >> bit) & 1) << (3 * bit + 2 - k)
    return code >> 7 if n <= 2**17 else code


@pytest.mark.parametrize("n", [1, 64, 65, 1023, 1025, 16384, 16385, 65536, 65537, 131072, 131073])
def test_primitive_order_is_the_stable_sort_of_the_codes(device, n):
    sc = workloads.scene(n, 1, 32, 32, scale_range=(0.005, 0.02), seed=n, device=device)
    f = fused.prepare(*sc.params(), sc.viewmats, sc.Ks, 32, 32, 1e-8, 3.0)
    perm = f.record_offsets[n + 1:].long()
    assert torch.equal(perm, torch.sort(_codes(sc.means, n), stable=True).indices)


# (primitives, views, width, height, tile edge): ranges of 64, 128 and 256
# records and more; tables of one tile, of up to 16 KB, and up to 40 KB with few
# waves (placed) and with many (sorted); more tiles than any table
SHAPES = [(1, 1, 16, 16, 16), (63, 2, 40, 24, 8), (65, 3, 8, 8, 8), (4097, 2, 96, 80, 16), (30011, 1, 517, 333, 16),
          (5000, 9, 300, 310, 16), (20000, 24, 200, 160, 8), (40003, 12, 250, 198, 16), (3000, 2, 600, 700, 16),
          (300, 70, 64, 64, 32)]


@pytest.mark.parametrize("n,views,w,h,tile", SHAPES)
def test_lists_hold_each_emission_once_in_its_tile(device, n, views, w, h, tile):
    sc = workloads.scene(n, views, h, w, scale_range=(0.005, 0.05), seed=n + tile, device=device)
    f = fused.prepare(*sc.params(), sc.viewmats, sc.Ks, w, h, 1e-8, 3.0, tile_size=tile)
    ntx, nty = -(-w // tile), -(-h // tile)
    perm = f.record_offsets[views * n + 1:].long()
    d = lambda x: x[perm].double() if x.shape[0] == n else x.double()  # noqa: E731
    covars, _ = ops.parameter_transform_fwd(d(sc.quats), d(sc.scales))
    m2, _, radii = ops.world_to_image_projection_fwd(d(sc.means), covars, sc.viewmats.double(), sc.Ks.double(), w, h,
                                                     1e-8, 3.0)
    counts, ids, flat = ops.isect_tiles(m2, radii, tile, ntx, nty)
    assert f.n_isects == ids.numel() == int(f.counters[0]) and int(f.counters[1]) == 0
    assert torch.equal(f.offsets, ops.isect_offset_encode(ids, views, ntx, nty))
    first = torch.zeros(views * n + 1, dtype=torch.long, device=device)
    first[1:] = torch.cumsum(counts.reshape(-1).long(), 0)
    assert torch.equal(f.record_offsets[: views * n + 1].long(), first)
    entries = f.packed[: f.n_isects * 8].view(torch.int32).reshape(-1, 2).long()
    assert torch.equal(torch.sort(entries[:, 1]).values, torch.arange(f.n_isects, device=device))
    # the operators' list holds the same records per tile
    key = ids.long() * (views * n)
    assert torch.equal(torch.sort(key + entries[:, 0]).values, torch.sort(key + flat.long()).values)
    # each emission index lies in its record's own range
    assert bool(((entries[:, 1] >= first[entries[:, 0]]) & (entries[:, 1] < first[entries[:, 0] + 1])).all())


@pytest.mark.parametrize("n,views,w,h", [(20011, 40, 520, 504), (3000, 3, 1100, 900), (3000, 2, 517, 333)])
def test_overflow_is_flagged_by_every_binning(device, n, views, w, h):
    sc = workloads.scene(n, views, h, w, scale_range=(0.005, 0.05), seed=4, device=device)
    f = fused.prepare(*sc.params(), sc.viewmats, sc.Ks, w, h, 1e-8, 3.0, capacity=1024, check=False)
    assert int(f.counters[1]) == 1 and int(f.counters[0]) > 1024
    assert not bool(fused.render(f, views, device).any())
