"""Bounds on what a thin primitive reaches: kernels that skip rows, octants, blocks
or columns against every voxel or pixel that a primitive's own form covers."""

import pytest
import torch

from r2splat_amd import fused, hip as ops, parity
from r2splat_amd.hip._wrapper import _isect_tiles_3d

pytestmark = pytest.mark.gpu

# ---------------------------------------------------------------------------
# voxel VJPs: discs of 40:1 to 100:1 tilted off the axes, half-axes of 15 to 60
# voxels, at beta 1/2. Both minors of such a form cancel, each by less than 1e-3,
# their product by more. The adjoint is 1 on the outer tenth of the support, so
# that a voxel of a dropped row shows in the sums. The reference sums the
# definition in double over the whole volume.
# ---------------------------------------------------------------------------
SIDE, DISCS = 96, 60


def _discs(seed):
    g = torch.Generator().manual_seed(seed)
    r = lambda *s: torch.rand(*s, generator=g, dtype=torch.float64)  # noqa: E731
    q, _ = torch.linalg.qr(r(DISCS, 3, 3) - 0.5)
    long = 15.0 + 45.0 * r(DISCS, 1)
    s = torch.cat([long / (40.0 + 60.0 * r(DISCS, 1)), long, long * (0.8 + 0.2 * r(DISCS, 1))], 1)
    P = q @ torch.diag_embed(s ** -2) @ q.transpose(1, 2)
    means = SIDE * (0.3 + 0.4 * r(DISCS, 3))
    return means, torch.stack([P[:, 0, 0], P[:, 0, 1], P[:, 0, 2], P[:, 1, 1], P[:, 1, 2], P[:, 2, 2]], 1)


def _disc_reference(mean, conic, beta, w):
    """(adjoint, sum v h^beta, sum v w h^beta log h) over the volume, in double."""
    axis = torch.arange(SIDE, device=mean.device, dtype=torch.float64) + 0.5
    z, y, x = torch.meshgrid(axis, axis, axis, indexing="ij")
    dx, dy, dz = x - mean[0], y - mean[1], z - mean[2]
    h = 1.0 - (conic[0] * dx * dx + conic[3] * dy * dy + conic[5] * dz * dz +
               2.0 * (conic[1] * dx * dy + conic[2] * dx * dz + conic[4] * dy * dz))
    shell = (h > 1e-4) & (h < 0.1)  # (the float32 form of the innermost 1e-4 carries no digits)
    vis = torch.where(shell, h, torch.ones_like(h)).pow(beta) * shell
    return shell.to(torch.float32), vis.sum(), (w * vis * torch.where(shell, h, torch.ones_like(h)).log()).sum()


@pytest.mark.parametrize("seed", [1, 2])
@pytest.mark.parametrize("kernel", ["fused", "operator", "operator, long lists"])
def test_voxel_vjps_of_thin_discs(device, kernel, seed):
    means, conics = (t.to(device) for t in _discs(seed))
    n = -(-SIDE // 8)
    radii = torch.full((1, 3), 4 * SIDE, dtype=torch.int32, device=device)
    for k in range(DISCS):
        mean, conic = means[k:k + 1].contiguous(), conics[k:k + 1].contiguous()
        if kernel == "fused":  # float32 weights; the form is double in both
            mean32 = mean.float()
            _, ids, flat, cum = _isect_tiles_3d(mean32, radii, 8, n, n, n)
            beta = torch.full((1,), 0.5, device=device)
            w = torch.full((1,), 0.7, device=device)
            v, v_w, v_beta = _disc_reference(means[k], conics[k], 0.5, float(w))
            state = dict(mapped=mean32, frame=torch.cat([mean, conic], 1).contiguous(), conics=conic.float(),
                         radii=radii, tile_cum=cum, isect_ids=ids, flatten_ids=flat)
            got = fused.voxel_vjp(state, w, beta, v, (SIDE, SIDE, SIDE))
            tol = 1e-5  # float32 sums of up to a few thousand terms of one sign
        else:
            # long lists for the size: four of the disc among primitives that are in no list
            copies, total = (4, 8000) if kernel != "operator" else (1, 1)
            mean, conic = mean.repeat(total, 1), conic.repeat(total, 1)
            reach = radii.repeat(total, 1)
            reach[copies:] = 0
            _, ids, flat = ops.isect_tiles_3d(mean, reach, 8, n, n, n)
            off = ops.isect_offset_encode_3d(ids, n, n, n)
            beta = torch.full((total,), 0.5, device=device, dtype=torch.float64)
            w = torch.full((total,), 0.7, device=device, dtype=torch.float64)
            v, v_w, v_beta = _disc_reference(means[k], conics[k], 0.5, 0.7)
            got = ops.beta_voxelize_to_voxels_bwd_per_gaussian(mean, conic, w, beta, off, ids, flat, v.double(), SIDE,
                                                               SIDE, SIDE, 8)
            tol = 1e-9
        assert ids.numel() == (4 if "long" in kernel else 1) * n ** 3
        for name, a, b in (("opacity", got[2][0], v_w), ("beta", got[3][0], v_beta)):
            assert abs(float(a) - float(b)) <= tol * abs(float(b)), (k, name, float(a), float(b))


# ---------------------------------------------------------------------------
# Beta rasterizer: needles of 1000:1 to 3000:1, hundreds of pixels long, whose end
# lies in the image. The 16-pixel forward walks 4 x 4 blocks and the backward
# segments of 8 columns, so each has a bound on columns beside the one on rows;
# the keep masks know the rows alone. A pixel is lit exactly where the forward's
# mask keeps the primitive, and an adjoint of one kept pixel reaches the density.
# ---------------------------------------------------------------------------
IMAGE, VIEWS = 160, 4096


def _needle(seed, device):
    g = torch.Generator().manual_seed(seed)
    r = lambda *s: torch.rand(*s, generator=g, dtype=torch.float64)  # noqa: E731
    f = 1.2 * IMAGE
    px = 2.5 / f  # world units of a pixel at the needle's depth
    half = 460.0
    theta, end = 6.2832 * r(VIEWS), IMAGE * (0.05 + 0.9 * r(VIEWS, 2)) - IMAGE / 2
    c, s = torch.cos(theta), torch.sin(theta)
    views = torch.zeros(VIEWS, 4, 4, dtype=torch.float64)
    views[:, 0, 0], views[:, 0, 1], views[:, 1, 0], views[:, 1, 1] = c, -s, s, c
    views[:, 2, 2] = views[:, 3, 3] = 1.0
    views[:, :2, 3] = (end - half * torch.stack([c, s], 1)) * px  # the needle's mean is the world origin
    views[:, 2, 3] = 2.5
    Ks = torch.tensor([[f, 0.0, IMAGE / 2], [0.0, f, IMAGE / 2], [0.0, 0.0, 1.0]], dtype=torch.float64)
    thin = half * px / (1000.0 + 2000.0 * float(r(1)))
    prims = [torch.zeros(1, 3), torch.tensor([[1.0, 0.0, 0.0, 0.0]]), torch.tensor([[half * px, thin, thin]]),
             torch.ones(1)]
    return ([t.to(device, torch.float32).contiguous() for t in prims],
            views.to(device, torch.float32), Ks.expand(VIEWS, 3, 3).to(device, torch.float32).contiguous())


def _pixels(table, words, device):
    """Which pixels [view, y, x] a keep mask keeps (one primitive)."""
    n, T = table.cam.numel(), table.tile
    bits = (words[:, :, None] >> torch.arange(32, device=device, dtype=torch.int32)) & 1
    e, p = bits.reshape(n, T * T).bool().nonzero(as_tuple=True)
    kept = torch.zeros(VIEWS, IMAGE, IMAGE, dtype=torch.bool, device=device)
    kept[table.cam[e], table.ty[e] * T + p // T, table.tx[e] * T + p % T] = True
    return kept


@pytest.mark.parametrize("seed", [1, 2, 3])
def test_beta_rasterizer_of_needles(device, seed):
    prims, views, Ks = _needle(seed, device)
    beta = torch.full((1,), 0.6, device=device)
    args = (*prims, views, Ks)
    image, fwd = fused.forward(*args, IMAGE, IMAGE, 1e-8, 1.0, beta=beta)
    table = parity.pair_table(fwd, VIEWS, 1)
    kept = _pixels(table, table.mask_fwd, device)
    assert int(kept.sum()) > VIEWS
    lit = image != 0
    strays, lost = int((lit & ~kept).sum()), int((kept & ~lit).sum())
    assert (strays, lost) == (0, 0)
    # the kept pixels nearest the needle's ends in x, one adjoint per view; views one by one
    both = kept & _pixels(table, table.mask_bwd, device) & (image > 1e-3)
    cols = both.any(1)
    first, last = cols.int().argmax(1), IMAGE - 1 - cols.flip(1).int().argmax(1)
    v = torch.zeros(1, IMAGE, IMAGE, device=device)
    for k in cols.any(1).nonzero().flatten().tolist()[:1500]:
        _, one = fused.forward(*prims, views[k:k + 1], Ks[k:k + 1], IMAGE, IMAGE, 1e-8, 1.0, beta=beta)
        for x in (int(first[k]), int(last[k])):
            y = int(both[k, :, x].int().argmax())
            v.zero_()[0, y, x] = 1.0
            grads = fused.backward(one, *prims, views[k:k + 1], Ks[k:k + 1], v)
            assert float(grads[3][0]) > 0.0, (k, y, x)
