"""The fused Beta rasterizer's 4 x 4 pixel blocks (forward) and 8-column row
segments (backward and list order) at their edges: supports smaller than a
pixel, of a few pixels and larger than a tile, image sides off the tile grid,
every binning path, against float64 over the kept pairs and the operators' lists."""

import pytest
import torch

import r2splat_amd
from oracle import splat as O
from r2splat_amd import fused, hip as ops, workloads
from r2splat_amd.parity import evaluate, fp64_scene, pair_table

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("uncertainty", [None, 0.1])
@pytest.mark.parametrize("n,views,h,w,scales", [(3000, 3, 49, 33, (0.002, 0.008)), (800, 2, 72, 56, (0.004, 0.04)),
                                                (120, 2, 65, 100, (0.05, 0.5)), (4000, 2, 530, 520, (0.003, 0.03))])
def test_beta_blocks_and_segments_against_float64(device, n, views, h, w, scales, uncertainty):
    sc = workloads.scene(n, views, h, w, scale_range=scales, seed=n, device=device, beta_range=(0.5, 4.0),
                         uncertainty_max=uncertainty)
    options = dict(beta=sc.beta, uncertainty=sc.uncertainty)
    out, ctx = r2splat_amd.rasterize_fwd(*sc.params(), sc.viewmats, sc.Ks, sc.image_size, **options)
    table = pair_table(ctx.buffers["fused"], views, n)
    image = out if uncertainty is None else out[0]
    g = torch.Generator(device=device).manual_seed(1)
    v = torch.randn(image.shape, generator=g, device=device) / image.numel()
    v_var = None if uncertainty is None else torch.randn(image.shape, generator=g, device=device) / image.numel()
    got = r2splat_amd.rasterize_bwd(ctx, v, v_var)
    sc64 = fp64_scene(*sc.params(), sc.viewmats, sc.Ks, sc.image_size, **options)
    kept = evaluate(table, sc64, "kept", v_image=v, **({} if v_var is None else dict(v_variance=v_var)))
    assert O.relative_error(image, kept.image) <= 1e-5
    for name in ("means", "quats", "scales", "densities", "beta"):
        err = O.relative_error(getattr(got, name), kept.grads[name])
        assert err <= 1e-4, f"{name}: {err:.2e}"


# small and large bin tables (placed) and more tiles than any table (sorted)
@pytest.mark.parametrize("n,views,w,h,tile", [(63, 2, 40, 24, 8), (40003, 12, 250, 198, 16), (5000, 1, 517, 333, 16),
                                              (3000, 2, 600, 700, 16), (300, 20, 64, 64, 32), (2000, 2, 1300, 1100, 32)])
def test_beta_lists_hold_each_emission_once_in_its_tile(device, n, views, w, h, tile):
    sc = workloads.scene(n, views, h, w, scale_range=(0.005, 0.05), seed=n + tile, device=device,
                         beta_range=(0.5, 4.0))
    f = fused.prepare(*sc.params(), sc.viewmats, sc.Ks, w, h, 1e-8, 1.0, tile_size=tile, beta=sc.beta)
    ntx, nty = -(-w // tile), -(-h // tile)
    perm = f.record_offsets[views * n + 1:].long()
    d = lambda x: x[perm].double() if x.shape[0] == n else x.double()  # noqa: E731
    covars, _ = ops.parameter_transform_fwd(d(sc.quats), d(sc.scales))
    m2, _, radii = ops.world_to_image_projection_fwd(d(sc.means), covars, sc.viewmats.double(), sc.Ks.double(), w, h,
                                                     1e-8, 1.0)
    _, ids, flat = ops.isect_tiles(m2, radii, tile, ntx, nty)
    assert f.n_isects == ids.numel()
    assert torch.equal(f.offsets, ops.isect_offset_encode(ids, views, ntx, nty))
    entries = f.packed[: f.n_isects * 8].view(torch.int32).reshape(-1, 2).long()
    assert torch.equal(torch.sort(entries[:, 1]).values, torch.arange(f.n_isects, device=device))
    key = ids.long() * (views * n)
    assert torch.equal(torch.sort(key + entries[:, 0]).values, torch.sort(key + flat.long()).values)
