"""The operator rasterizer's kernels for 8, 16 and 32 pixel tiles (rows a primitive
does not reach skipped; tiles split over workgroups in small launches) and the
operator voxelizer's for 8^3 tiles against their general kernels: every primitive
is binned to every tile, so the tile edge changes nothing but the kernel."""

import pytest
import torch

from oracle import splat as O
from r2splat_amd import hip as ops

pytestmark = pytest.mark.gpu


def _case(device, dtype, C, N, W, H, seed, beta, var):
    g = torch.Generator().manual_seed(seed)
    r = lambda *s: torch.rand(*s, generator=g, dtype=torch.float64)  # noqa: E731
    means = torch.stack([r(C, N) * (W + 20) - 10, r(C, N) * (H + 20) - 10], -1)
    theta, s1, s2 = r(C, N) * 3.1416, torch.exp(r(C, N) * 4 - 1.5), torch.exp(r(C, N) * 4 - 1.5)
    c, s = torch.cos(theta), torch.sin(theta)
    conics = torch.stack([c * c / s1**2 + s * s / s2**2, c * s * (1 / s1**2 - 1 / s2**2),
                          s * s / s1**2 + c * c / s2**2], -1)
    opac, mus = r(C, N), r(C, N) + 0.05
    opac[:, :2] = 1e-7  # never above the cut-off
    if N > 6:
        conics[:, 2] = torch.tensor([0.0, 0.0, 0.0])  # flat: reaches every pixel
        conics[:, 3] = torch.tensor([1.0, 1.5, 1.0])  # indefinite
    out = [t.to(device, dtype) for t in (means, conics, opac, mus)]
    betas = (0.6 + 3 * r(C, N)).to(device, dtype) if beta else None
    unc = (0.1 * r(N)).to(device, dtype) if var else None
    v = (r(C, H, W) - 0.5).to(device, dtype)
    vv = (r(C, H, W) - 0.5).to(device, dtype) if var else None
    return out, betas, unc, v, vv


def _run(case, W, H, T, listed=None):
    """Every primitive in every tile, or the first `listed` of each camera."""
    (means, conics, opac, mus), betas, unc, v, vv = case
    C, N = opac.shape
    listed = N if listed is None else listed
    nx, ny = -(-W // T), -(-H // T)
    radii = torch.zeros((C, N, 2), dtype=torch.int32, device=means.device)
    radii[:, :listed] = 4 * (W + H)
    _, ids, flat = ops.isect_tiles(means, radii, T, nx, ny)
    assert ids.numel() == C * listed * nx * ny
    off = ops.isect_offset_encode(ids, C, nx, ny)
    args = (means, conics, opac, mus) + (() if betas is None else (betas,))
    pre = "" if betas is None else "beta_"
    if unc is None:
        img = (getattr(ops, pre + "rasterize_to_pixels_fwd")(*args, off, flat, W, H, T),)
        grads = getattr(ops, pre + "rasterize_to_pixels_bwd_per_gaussian")(*args, off, ids, flat, v, W, H, T, False)
    else:
        img = getattr(ops, pre + "rasterize_to_pixels_mean_var_fwd")(*args, unc, off, flat, W, H, T)
        grads = getattr(ops, pre + "rasterize_to_pixels_mean_var_bwd_per_gaussian")(
            *args, off, ids, flat, v, vv, unc, False, W, H, T, False)
    return img, [g for g in grads if g is not None]


# (cameras, primitives, width, height, tile): launches that are split and that
# are not, more than 2^19 intersections, ragged edges, fewer records than a wave
SHAPES = [(2, 7, 40, 24, 8), (12, 100, 200, 160, 8), (1, 70, 61, 47, 16), (36, 9, 190, 160, 16), (2, 300, 70, 33, 32),
          (33, 20, 512, 384, 32)]


@pytest.mark.parametrize("dtype", [torch.float32, torch.float64])
@pytest.mark.parametrize("beta,var", [(False, False), (False, True), (True, False), (True, True)])
@pytest.mark.parametrize("C,N,W,H,T", SHAPES)
def test_row_kernels_match_the_general_kernel(device, C, N, W, H, T, beta, var, dtype):
    case = _case(device, dtype, C, N, W, H, C + N, beta, var)
    _compare(lambda c, t: _run(c, W, H, t), case, T, 10)


# A small launch of short lists takes the general kernel: these are of the sizes, for
# primitives that fill their tiles, from which the VJP's row kernels are chosen.
@pytest.mark.parametrize("dtype", [torch.float32, torch.float64])
@pytest.mark.parametrize("beta,var", [(False, False), (False, True), (True, False), (True, True)])
@pytest.mark.parametrize("C,N,W,H,T", [(2, 150, 77, 90, 8), (2, 600, 200, 157, 16), (3, 1000, 320, 319, 32)])
def test_row_kernels_of_long_lists(device, C, N, W, H, T, beta, var, dtype):
    case = _case(device, dtype, C, N, W, H, C + N, beta, var)
    _compare(lambda c, t: _run(c, W, H, t), case, T, 10)


@pytest.mark.parametrize("dtype", [torch.float32, torch.float64])
@pytest.mark.parametrize("beta,var", [(False, True), (True, True)])
@pytest.mark.parametrize("W,H,T", [(200, 160, 8), (390, 319, 16), (799, 620, 32)])
def test_forward_row_kernels_of_many_tiles(device, W, H, T, beta, var, dtype):
    """4500 tiles, more than the forward splits over workgroups; primitives that stand
    in no list beside the 50 of each camera, so that lists are long for the footprints."""
    C, listed = 9, 50
    case = _case(device, dtype, C, listed * 500, W, H, T, beta, var)
    _compare(lambda c, t: (_run(c, W, H, t, listed)[0], []), case, T, 10)


def _compare(run, case, tile, other):
    got, general = run(case, tile), run(case, other)
    dtype = case[0][0].dtype
    assert len(got[1]) == len(general[1])
    if dtype == torch.float64:  # the same terms summed in another order
        for tol, new, old in ((1e-12, got[0], general[0]), (1e-11, got[1], general[1])):
            for k, (a, b) in enumerate(zip(new, old)):
                assert O.relative_error(a, b) <= tol, k
        return
    # float32 forms of thin footprints cancel, so both kernels are a few roundings
    # of terms far above the exponent away from float64: as near as the general one
    wide = [t.double() for t in case[0]], *(None if t is None else t.double() for t in case[1:])
    exact = run(wide, other)
    for tol, new, old, ref in ((1e-5, got[0], general[0], exact[0]), (1e-4, got[1], general[1], exact[1])):
        for k, (a, b, r) in enumerate(zip(new, old, ref)):
            e_new, e_old = O.relative_error(a.double(), r), O.relative_error(b.double(), r)
            print(f"output {k}: {e_new:.2e}, general kernel {e_old:.2e}")
            assert e_new <= tol + 2.0 * e_old, k


def _voxel_case(device, dtype, N, dims, seed, beta, var):
    g = torch.Generator().manual_seed(seed)
    r = lambda *s: torch.rand(*s, generator=g, dtype=torch.float64)  # noqa: E731
    means = r(N, 3) * (torch.tensor(dims, dtype=torch.float64) + 6) - 3
    q, _ = torch.linalg.qr(r(N, 3, 3) - 0.5)
    m = q @ torch.diag_embed(torch.exp(4 - 8 * r(N, 3)) * 0.2) @ q.transpose(1, 2)
    conics = torch.stack([m[:, 0, 0], m[:, 0, 1], m[:, 0, 2], m[:, 1, 1], m[:, 1, 2], m[:, 2, 2]], -1)
    opac = r(N)
    opac[:2] = 1e-8
    if N > 6:
        conics[2] = 0.0
        conics[3] = torch.tensor([1.0, 1.5, 0.2, 1.0, 0.1, 1.0])  # indefinite
    out = [t.to(device, dtype) for t in (means, conics, opac)]
    betas = (0.6 + 3 * r(N)).to(device, dtype) if beta else None
    unc = (0.1 * r(N)).to(device, dtype) if var else None
    v, vv = ((r(*dims[::-1]) - 0.5).to(device, dtype) for _ in range(2))
    return out, betas, unc, v, vv if var else None


def _voxel_run(case, dims, T):
    (means, conics, opac), betas, unc, v, vv = case
    n = [-(-d // T) for d in dims]
    radii = torch.full((opac.numel(), 3), 4 * sum(dims), dtype=torch.int32, device=means.device)
    _, ids, flat = ops.isect_tiles_3d(means, radii, T, *n)
    off = ops.isect_offset_encode_3d(ids, *n)
    args = (means, conics, opac) + (() if betas is None else (betas,))
    pre = "" if betas is None else "beta_"
    if unc is None:
        img = (getattr(ops, pre + "voxelize_to_voxels_fwd")(*args, off, flat, *dims, T),)
        grads = getattr(ops, pre + "voxelize_to_voxels_bwd_per_gaussian")(*args, off, ids, flat, v, *dims, T)
    else:
        img = getattr(ops, pre + "voxelize_to_voxels_mean_var_fwd")(*args, unc, off, flat, *dims, T)
        grads = getattr(ops, pre + "voxelize_to_voxels_mean_var_bwd_per_gaussian")(
            *args, off, ids, flat, v, vv, unc, False, *dims, T)
    return img, [g for g in grads if g is not None]


@pytest.mark.parametrize("dtype", [torch.float32, torch.float64])
@pytest.mark.parametrize("beta,var", [(False, False), (False, True), (True, False), (True, True)])
@pytest.mark.parametrize("N,dims", [(5, (16, 8, 9)), (90, (37, 21, 30)), (1100, (64, 64, 60))])
def test_voxel_8_tiles_match_the_general_kernel(device, N, dims, beta, var, dtype):
    case = _voxel_case(device, dtype, N, dims, N, beta, var)
    moments = dtype == torch.float32 and not (beta or var)  # its VJP is another kernel

    def run(c, t):
        img, grads = _voxel_run(c, dims, t)
        return img, [] if moments else grads

    _compare(run, case, 8, 7)


@pytest.mark.parametrize("dtype", [torch.float32, torch.float64])
@pytest.mark.parametrize("beta,var", [(False, False), (False, True), (True, False), (True, True)])
def test_voxel_8_tiles_of_long_lists(device, beta, var, dtype):
    """Fewer than 2^19 intersections, from which the kernels take the longer chunk."""
    N, dims = 420, (40, 47, 37)
    case = _voxel_case(device, dtype, N, dims, N, beta, var)
    moments = dtype == torch.float32 and not (beta or var)  # its VJP is another kernel

    def run(c, t):
        img, grads = _voxel_run(c, dims, t)
        return img, [] if moments else grads

    _compare(run, case, 8, 7)


def _same_marks(got, general, image, what):
    """Images: NaN and either infinity in the same places; gradients: the same values
    finite (an infinite sum may be infinite or NaN by its order). The finite values
    are one sum in two orders."""
    for k, (a, b) in enumerate(zip(got, general)):
        for mark in (torch.isnan, torch.isposinf, torch.isneginf) if image else (torch.isfinite,):
            assert torch.equal(mark(a), mark(b)), (*what, k, int(mark(a).sum()), int(mark(b).sum()))
        x, y = a[b.isfinite()], b[b.isfinite()]
        if y.numel():
            assert float((x - y).abs().max()) <= 1e-11 * float(y.abs().max()), (*what, k)


NONFINITE = [float("nan"), float("inf"), float("-inf")]


@pytest.mark.parametrize("beta,var", [(False, True), (True, True)])
@pytest.mark.parametrize("T,N,pad", [(8, 20, 0), (16, 20, 0), (32, 20, 0),
                                     (8, 20, 2000), (16, 30, 500), (32, 1400, 8000)])  # padded: long lists for the size
def test_row_kernels_keep_nonfinite_parameters_to_their_pairs(device, T, N, pad, beta, var):
    """A primitive with a NaN or an infinity marks the pixels and gradients that the
    general kernel marks: those of its own pairs past the cut-off. `pad` primitives
    stand in no list, as off-screen ones do."""
    W, H = 70, 45
    for value in NONFINITE:
        for field in ("mean", "conic a", "conic b", "opacity", "mu", "beta", "uncertainty"):
            if field == "beta" and not beta:
                continue
            (means, conics, opac, mus), betas, unc, v, vv = _case(device, torch.float64, 1, N + pad, W, H, 11, beta, var)
            target = {"mean": means[0, 7], "conic a": conics[0, 7], "conic b": conics[0, 7, 1:], "opacity": opac[0, 7:],
                      "mu": mus[0, 7:], "beta": None if betas is None else betas[0, 7:], "uncertainty": unc[7:]}[field]
            target[0] = value
            case = ((means, conics, opac, mus), betas, unc, v, vv)
            (img, grads), (ref, expected) = (_run_lists(case, W, H, t, N) for t in (T, 10))
            _same_marks(img, ref, True, (value, field, "image"))
            _same_marks(grads, expected, False, (value, field, "gradient"))


def _run_lists(case, W, H, T, N):
    """_run with the first N primitives in every tile whatever their means hold."""
    (means, conics, opac, mus), betas, unc, v, vv = case
    C = opac.shape[0]
    nt = -(-W // T) * -(-H // T)
    dev = means.device
    flat = torch.arange(N, dtype=torch.int32, device=dev).repeat(nt)
    ids = torch.arange(nt, device=dev).repeat_interleave(N)
    off = ops.isect_offset_encode(ids, C, -(-W // T), -(-H // T))
    args = (means, conics, opac, mus) + (() if betas is None else (betas,))
    pre = "" if betas is None else "beta_"
    img = getattr(ops, pre + "rasterize_to_pixels_mean_var_fwd")(*args, unc, off, flat, W, H, T)
    grads = getattr(ops, pre + "rasterize_to_pixels_mean_var_bwd_per_gaussian")(
        *args, off, ids, flat, v, vv, unc, False, W, H, T, False)
    return img, [g for g in grads if g is not None]


@pytest.mark.parametrize("beta", [False, True])
@pytest.mark.parametrize("N,pad", [(20, 0), (120, 6000)])  # padded: long lists for the size
def test_voxel_8_tiles_keep_nonfinite_parameters_to_their_pairs(device, N, pad, beta):
    dims = (21, 17, 30)
    for value in NONFINITE:
        for field in ("mean", "conic xx", "conic xy", "opacity", "beta", "uncertainty"):
            if field == "beta" and not beta:
                continue
            (means, conics, opac), betas, unc, v, vv = _voxel_case(device, torch.float64, N + pad, dims, 11, beta, True)
            target = {"mean": means[7], "conic xx": conics[7], "conic xy": conics[7, 1:], "opacity": opac[7:],
                      "beta": None if betas is None else betas[7:], "uncertainty": unc[7:]}[field]
            target[0] = value
            args = (means, conics, opac) + (() if betas is None else (betas,))
            pre = "beta_" if beta else ""
            out = []
            for T in (8, 7):
                n = [-(-d // T) for d in dims]
                nt = n[0] * n[1] * n[2]
                flat = torch.arange(N, dtype=torch.int32, device=device).repeat(nt)
                ids = torch.arange(nt, device=device).repeat_interleave(N)
                off = ops.isect_offset_encode_3d(ids, *n)
                img = getattr(ops, pre + "voxelize_to_voxels_mean_var_fwd")(*args, unc, off, flat, *dims, T)
                grads = getattr(ops, pre + "voxelize_to_voxels_mean_var_bwd_per_gaussian")(
                    *args, off, ids, flat, v, vv, unc, False, *dims, T)
                out.append((img, [g for g in grads if g is not None]))
            _same_marks(out[0][0], out[1][0], True, (value, field, "volume"))
            _same_marks(out[0][1], out[1][1], False, (value, field, "gradient"))


@pytest.mark.parametrize("beta", [False, True])
def test_float32_moments_show_a_nan_mean(device, beta):
    dims, N = (21, 17, 30), 20
    (means, conics, opac), betas, _, v, _ = _voxel_case(device, torch.float32, N, dims, 11, beta, False)
    means[7, 1] = float("nan")
    n = [-(-d // 8) for d in dims]
    nt = n[0] * n[1] * n[2]
    flat = torch.arange(N, dtype=torch.int32, device=device).repeat(nt)
    ids = torch.arange(nt, device=device).repeat_interleave(N)
    off = ops.isect_offset_encode_3d(ids, *n)
    args = (means, conics, opac) + (() if betas is None else (betas,))
    grads = getattr(ops, ("beta_" if beta else "") + "voxelize_to_voxels_bwd_per_gaussian")(*args, off, ids, flat, v,
                                                                                            *dims, 8)
    for k, g in enumerate(grads[:2]):  # mean and conic
        rows = g.isnan().any(-1)
        assert rows.nonzero().flatten().tolist() == [7], k


@pytest.mark.parametrize("beta,var", [(False, False), (False, True), (True, False), (True, True)])
@pytest.mark.parametrize("T", [8, 16, 32])
def test_float32_vjp_sums_are_as_near_as_the_general_kernels(device, T, beta, var):
    """Round footprints, whose terms carry no cancellation: what is left is how the
    VJP adds them. The root mean square error over 1200 primitives and four scenes
    varies by a few percent (the largest error by half); a quarter more than the
    general kernel's is a longer chain of float sums."""
    C, N, W, H = 3, 400, 150, 110
    total = 8000 if T == 32 else N  # of which N in the lists: the row kernel from 24k intersections
    new, old = 0.0, 0.0
    for seed in range(4):
        g = torch.Generator().manual_seed(seed)
        r = lambda *s: torch.rand(*s, generator=g, dtype=torch.float64)  # noqa: E731
        means = torch.stack([r(C, N) * W, r(C, N) * H], -1)
        s = 1.5 + 4.5 * r(C, N)
        conics = torch.stack([s**-2, 0.1 * s**-2, s**-2], -1)
        prims = [t.to(device, torch.float32) for t in (means, conics, r(C, N), r(C, N) + 0.05)]
        betas = (0.6 + 3 * r(C, N)).to(device, torch.float32) if beta else None
        unc = (0.1 * r(N)).to(device, torch.float32) if var else None
        v, vv = ((r(C, H, W) - 0.5).to(device, torch.float32) for _ in range(2))
        extra = total - N
        prims = [torch.cat([t, t[:, :1].expand(C, extra, *t.shape[2:])], 1).contiguous() for t in prims]
        betas = None if betas is None else torch.cat([betas, betas[:, :1].expand(C, extra)], 1).contiguous()
        unc = None if unc is None else torch.cat([unc, unc[:1].expand(extra)]).contiguous()
        case = (prims, betas, unc, v, vv if var else None)
        wide = [t.double() for t in prims], *(None if t is None else t.double() for t in case[1:])
        exact = _run(wide, W, H, 10, N)[1]
        errors = lambda tile: torch.tensor(  # noqa: E731
            [float((a.double() - b).norm() / b.norm()) for a, b in zip(_run(case, W, H, tile, N)[1], exact)])
        new, old = new + errors(T), old + errors(10)
    assert bool((new <= 1.25 * old).all()), (new / old).tolist()


def _vjp_time(run):
    """Least of ten timed calls after one untimed, in ms."""
    run()
    times = []
    for _ in range(10):
        start, end = (torch.cuda.Event(enable_timing=True) for _ in range(2))
        start.record()
        run()
        end.record()
        end.synchronize()
        times.append(start.elapsed_time(end))
    return min(times)


@pytest.mark.parametrize("kind", ["raster", "voxel"])
def test_vjps_of_sparse_lists_take_no_lane_per_intersection(device, kind):
    """A few hundred Beta primitives that fill their tiles, in float64: a wave each takes
    some 30 us beside the call's own, a lane each 2 to 5 ms. The general kernel of a tile
    edge that has no other is the measure; four times it is far from both."""
    if kind == "raster":
        case, W, H = _case(device, torch.float64, 1, 8, 256, 256, 5, True, False), 256, 256
        run = lambda T: _run(case, W, H, T)  # noqa: E731
        tiles = (32, 31)
    else:
        case, dims = _voxel_case(device, torch.float64, 8, (48, 48, 48), 5, True, False), (48, 48, 48)
        run = lambda T: _voxel_run(case, dims, T)  # noqa: E731
        tiles = (8, 7)
    new, general = (_vjp_time(lambda: run(T)) for T in tiles)
    assert new <= 4.0 * general, (new, general)
