"""Fused voxel kernels where their work division can go wrong: one
intersection, chunks that end inside a tile and that span many tiles, both
chunk sizes, volumes off the tile grid, needle-shaped primitives (whose row
bound does not apply), supports smaller than a voxel; against the float64
operators on the same tile lists (the lists come from the float32 mapping,
whose footprint radii differ from float64's for needles) and the same
double-precision frame."""

import pytest
import torch

from oracle import splat as O
from r2splat_amd import explicit, fused, hip as ops, workloads

pytestmark = pytest.mark.gpu

# (primitives, volume shape, scale range)
CASES = [(1, (8, 8, 8), (0.1, 0.2)), (300, (9, 17, 23), (0.02, 0.2)), (3000, (40, 33, 48), (0.004, 0.01)),
         (30000, (64, 56, 64), (0.02, 0.05))]
# axes up to 600 : 1, for Beta primitives, whose forms are evaluated in double (a
# Gaussian's float32 form of this condition carries no digits to compare)
NEEDLES = (700, (24, 40, 16), (0.0005, 0.3))


@pytest.mark.parametrize("n,shape,scales,beta,var",
                         [(*case, beta, var) for case in CASES for beta in (False, True) for var in (False, True)] +
                         [(*NEEDLES, True, var) for var in (False, True)])
def test_fused_voxels_match_float64(device, n, shape, scales, beta, var):
    sc = workloads.scene(n, 1, 8, 8, scale_range=scales, seed=n, device=device,
                         beta_range=(0.5, 4.0) if beta else None, uncertainty_max=0.1 if var else None)
    g = torch.Generator(device=device).manual_seed(n)
    v = torch.randn(shape, generator=g, device=device)
    vv = torch.randn(shape, generator=g, device=device) if var else None
    depth, height, width = shape
    dims = (width, height, depth)
    one, zero = torch.ones(3, device=device), torch.zeros(3, device=device)
    vol = dict(extent=one, center=zero, extent64=one.double(), center64=zero.double())
    b = explicit._voxel_state((*sc.params(), sc.beta, sc.uncertainty), vol, shape, 1e-8, 1.0 if beta else 3.0)
    out = fused.voxel_render(b, sc.densities, sc.beta, dims, uncertainty=sc.uncertainty)
    grads = fused.voxel_vjp(b, sc.densities, sc.beta, v, dims, uncertainty=sc.uncertainty, v_variance=vv)

    d = lambda t: t.double().contiguous()  # noqa: E731
    args = [d(b["frame"][:, :3]), d(b["frame"][:, 3:]), d(sc.densities)] + ([d(sc.beta)] if beta else [])
    prefix = "beta_" if beta else ""
    if var:
        ref = getattr(ops, prefix + "voxelize_to_voxels_mean_var_fwd")(
            *args, d(sc.uncertainty), b["offsets"], b["flatten_ids"], *dims, 8)
        expected = getattr(ops, prefix + "voxelize_to_voxels_mean_var_bwd_per_gaussian")(
            *args, b["offsets"], b["isect_ids"], b["flatten_ids"], d(v), d(vv), d(sc.uncertainty), False, *dims, 8)
    else:
        ref = (getattr(ops, prefix + "voxelize_to_voxels_fwd")(*args, b["offsets"], b["flatten_ids"], *dims, 8),)
        out = (out,)
        expected = getattr(ops, prefix + "voxelize_to_voxels_bwd_per_gaussian")(
            *args, b["offsets"], b["isect_ids"], b["flatten_ids"], d(v), *dims, 8)
    for x, y in zip(out, ref):
        assert O.relative_error(x, y) <= 1e-5
    assert len(grads) == len(expected)
    for k, (x, y) in enumerate(zip(grads, expected)):
        assert O.relative_error(x, y) <= 1e-4, k
