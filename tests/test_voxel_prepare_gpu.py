"""The voxel prepare and parameter VJP calls against the operators they
stand for (bitwise), and the exclusive scan around its 16-byte runs."""

import pytest
import torch

from r2splat_amd import explicit, fused, hip as ops, profiling, workloads
from r2splat_amd.hip import _backend as be, _wrapper

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("dtype", [torch.float32, torch.float64])
@pytest.mark.parametrize("n,dims,scales", [(1, (8, 8, 8), (0.05, 0.1)), (257, (51, 62, 45), (0.01, 0.08)),
                                           (5000, (20, 9, 33), (0.001, 0.5)), (70_001, (130, 64, 72), (0.005, 0.05)),
                                           (300, (16, 16, 16), (1e-9, 2e-9))])
def test_voxel_prepare_equals_the_operators(device, n, dims, scales, dtype):
    sc = workloads.scene(n, 1, 8, 8, scale_range=scales, seed=n, device=device, dtype=dtype)
    means, quats, scls = sc.means * 1.3, sc.quats, sc.scales  # some primitives outside the volume
    extent64 = torch.tensor([1.0, 0.9, 1.1], dtype=torch.float64, device=device)
    center64 = torch.tensor([0.0, 0.05, -0.1], dtype=torch.float64, device=device)
    extent, center = extent64.to(dtype), center64.to(dtype)
    tiles = tuple(-(-d // 8) for d in dims)
    got = _wrapper.voxel_prepare(means, quats, scls, extent, center, extent64, center64, dims, 1e-8, 3.0, 8, tiles)
    covars, largest = ops.parameter_transform_fwd(quats, scls)
    mapped, conics, radii = ops.world_to_volume_mapping_fwd(means, covars, largest, extent, center, *dims, 1e-8, 3.0)
    _, ids, flat, cum = _wrapper._isect_tiles_3d(mapped, radii, 8, *tiles)
    expected = dict(covars=covars, mapped=mapped, conics=conics, radii=radii, tile_cum=cum, isect_ids=ids,
                    flatten_ids=flat, offsets=ops.isect_offset_encode_3d(ids, *tiles))
    if dtype == torch.float32:
        expected["frame"] = fused.voxel_frame(means, quats, scls, extent64, center64, dims, 1e-8)
    assert got.keys() == expected.keys()
    for name, value in expected.items():
        assert torch.equal(got[name], value), name
    g = torch.Generator(device=device).manual_seed(2)
    v_mapped = torch.randn(n, 3, generator=g, device=device, dtype=dtype)
    v_conics = torch.randn(n, 6, generator=g, device=device, dtype=dtype)
    v_means, v_covars = ops.world_to_volume_mapping_bwd(means, covars, extent, center, *dims, 1e-8, v_mapped, v_conics)
    want = (v_means, *ops.parameter_transform_bwd(quats, scls, v_covars))
    for a, b in zip(_wrapper.voxel_param_vjp(means, quats, scls, covars, extent, center, dims, 1e-8, v_mapped,
                                              v_conics), want):
        assert torch.equal(a, b)


def test_voxelize_of_primitives_that_reach_no_tile(device):
    sc = workloads.scene(50, 1, 8, 8, scale_range=(0.01, 0.02), seed=1, device=device)
    out, ctx = explicit.voxelize_fwd(sc.means + 5.0, *sc.params()[1:], (9, 10, 11), volume_extent=(1.0, 1.0, 1.0))
    assert not bool(out.any())
    assert not bool(explicit.voxelize_bwd(ctx, torch.ones_like(out)).densities.any())


@pytest.mark.parametrize("dtype", [torch.float32, torch.float64])
@pytest.mark.parametrize("backend", ["fused", "ops"])
def test_voxelize_reports_its_stages(device, monkeypatch, backend, dtype):
    sc = workloads.scene(50, 1, 8, 8, scale_range=(0.05, 0.1), seed=1, device=device, dtype=dtype)
    monkeypatch.setattr(explicit, "BACKEND", backend)
    profiling.reset()
    profiling.enable()
    try:
        out, ctx = explicit.voxelize_fwd(*sc.params(), (9, 10, 11), volume_extent=(1.0, 1.0, 1.0))
        explicit.voxelize_bwd(ctx, torch.ones_like(out))
        stages = set(profiling.collect())
    finally:
        profiling.enable(False)
        profiling.reset()
    assert {"voxel_map", "voxel_bin", "voxel_map_bwd"} <= stages


# a one-launch scan of either kind and a scan of levels, whole and cut 16-byte runs
@pytest.mark.parametrize("n", [1, 7, 8, 2047, 2048, 2049, 16383, 16384, 16385, 100_003])
def test_exclusive_scan_of_tile_counts(device, n):
    g = torch.Generator(device=device).manual_seed(n)
    radii = torch.randint(1, 12, (n, 3), generator=g, device=device, dtype=torch.int32)
    mapped = torch.rand(n, 3, generator=g, device=device) * 24.0
    tiles, ids, _, cum = _wrapper._isect_tiles_3d(mapped, radii, 8, 3, 3, 3)
    assert int(cum[0]) == 0 and torch.equal(cum[1:].long(), torch.cumsum(tiles.long(), 0))
    assert ids.numel() == int(cum[-1])
    assert be.lib().r2s_scan_workspace_bytes(n) > 0
