"""Volume and image loss kernels at the edges of their packing: row lengths
that are and are not a multiple of a 16-byte pack, pointers off that boundary,
plane counts around the gradient's march, and more packs than one sweep."""

import pytest
import torch

from oracle import splat as O
from r2splat_amd import hip as ops
from r2splat_amd.hip import _backend as be

pytestmark = pytest.mark.gpu

SHAPES = [(1, 1, 1, 1), (1, 8, 2, 4), (2, 9, 3, 8), (1, 17, 5, 3), (3, 7, 1, 12), (1, 130, 128, 132)]


def _place(x, device, offset):
    """x on the device, its first element `offset` elements past an allocation's start."""
    flat = torch.empty(x.numel() + offset, dtype=x.dtype, device=device)
    out = flat[offset:].view(x.shape)
    out.copy_(x)
    return out


@pytest.mark.parametrize("dtype", [torch.float32, torch.float64])
@pytest.mark.parametrize("offset", [0, 1])
@pytest.mark.parametrize("shape", SHAPES)
def test_tv_losses_at_pack_edges(shape, offset, dtype):
    device = torch.device("cuda:0")
    g = torch.Generator().manual_seed(sum(shape) + offset)
    vol = torch.randn(*shape, generator=g, dtype=torch.float64).to(dtype)
    ref = vol.double().requires_grad_()
    x = _place(vol, device, offset)
    one = torch.ones(1, device=device, dtype=dtype)
    # one rounding per operation of a short chain; the sums of n terms of one
    # sign in chains of at most 512 partial sums
    t = 2e-6 if dtype == torch.float32 else 1e-12
    for fwd, bwd, oracle in ((ops.volume_loss_fwd, ops.volume_loss_bwd, O.volume_tv(ref)),
                             (ops.volume_loss_iso_fwd, ops.volume_loss_iso_bwd, O.volume_tv_iso(ref, 1e-8))):
        (grad,) = torch.autograd.grad(oracle, ref)
        _, tv, tv_map = fwd(x, 1.0)
        assert abs(tv.item() - oracle.item()) <= t * abs(oracle.item())
        n = max(sum(s1 for s1 in _edge_counts(shape)), 1) if fwd is ops.volume_loss_fwd else vol.numel()
        assert abs(tv_map.double().sum().item() / n - oracle.item()) <= t * abs(oracle.item())
        got = bwd(x, one, 1.0)
        assert O.relative_error(got, grad) <= 5 * t


def _edge_counts(shape):
    B, D, H, W = shape
    return B * (D - 1) * H * W, B * D * (H - 1) * W, B * D * H * (W - 1)


@pytest.mark.parametrize("dtype", [torch.float32, torch.float64])
@pytest.mark.parametrize("n,offset", [(1, 0), (4, 0), (1023, 0), (4096, 1), (2_200_000, 0)])
def test_image_l1_at_pack_edges(n, offset, dtype):
    device = torch.device("cuda:0")
    g = torch.Generator().manual_seed(n)
    p = torch.randn(1, 1, n, generator=g, dtype=torch.float64).to(dtype)
    q = torch.randn(1, 1, n, generator=g, dtype=torch.float64).to(dtype)
    _, l1, l1_map = ops.image_loss_l1_fwd(_place(p, device, offset), _place(q, device, offset), 1.0)
    expected = (p - q).abs()
    assert torch.equal(l1_map.cpu(), expected)
    t = 2e-6 if dtype == torch.float32 else 1e-12
    assert abs(l1.item() - expected.double().mean().item()) <= t * expected.double().mean().item()


# rows of fewer, as many and more packs than a workgroup has threads, and workgroups
# whose threads lie in several plane chunks of different lengths
@pytest.mark.parametrize("dtype", [torch.float32, torch.float64])
@pytest.mark.parametrize("shape", [(1, 9, 7, 20), (2, 3, 33, 6), (1, 20, 3, 2048), (1, 10, 2, 2052), (1, 11, 5, 1031),
                                   (3, 17, 2, 4)])
def test_isotropic_gradient_where_threads_share_terms(shape, dtype):
    device = torch.device("cuda:0")
    g = torch.Generator().manual_seed(sum(shape))
    vol = torch.randn(*shape, generator=g, dtype=torch.float64).to(dtype)
    ref = vol.double().requires_grad_()
    (grad,) = torch.autograd.grad(O.volume_tv_iso(ref, 1e-8), ref)
    got = ops.volume_loss_iso_bwd(vol.to(device), torch.ones(1, device=device, dtype=dtype), 1.0)
    t = 1e-5 if dtype == torch.float32 else 5e-12  # as above: five roundings of a short chain
    assert O.relative_error(got, grad) <= t


@pytest.mark.parametrize("dtype", [torch.float32, torch.float64])
@pytest.mark.parametrize("shape", [(1, 1, 1, 1), (2, 9, 3, 8), (3, 7, 5, 13), (1, 130, 128, 132)])
def test_plain_sums_of_the_c_entries(shape, dtype):
    """r2s_volume_tv_fwd, r2s_volume_tv_iso_fwd and r2s_image_l1_fwd, which add
    their workgroups' sums by atomics: one workgroup and several, twice into one
    result, against the maps they leave and the operators' maps."""
    device = torch.device("cuda:0")
    g = torch.Generator().manual_seed(sum(shape))
    x, y = (torch.randn(*shape, generator=g, dtype=torch.float64).to(device, dtype) for _ in range(2))
    code, stream = be.dtype_code(dtype), be.stream_of(device)
    # sums of n positive terms: chains of at most 512 in the dtype, then in double;
    # one rounding to the dtype for each of at most 512 workgroups
    t = 5e-5 if dtype == torch.float32 else 1e-12
    calls = (("r2s_volume_tv_fwd", (x.data_ptr(), *shape), ops.volume_loss_fwd(x, 1.0)[2]),
             ("r2s_volume_tv_iso_fwd", (x.data_ptr(), *shape, 1e-8), ops.volume_loss_iso_fwd(x, 1.0)[2]),
             ("r2s_image_l1_fwd", (x.data_ptr(), y.data_ptr(), x.numel()),
              ops.image_loss_l1_fwd(x.flatten(0, 1), y.flatten(0, 1), 1.0)[2]))
    for name, args, expected in calls:
        out, total = torch.empty_like(x), torch.full((1,), 7.0, device=device, dtype=dtype)
        for _ in range(2):
            be.call(name, code, *args, out.data_ptr(), total.data_ptr(), stream)
            assert torch.equal(out.flatten(), expected.flatten())
            exact = out.double().sum().item()
            assert abs(total.item() - exact) <= t * exact
