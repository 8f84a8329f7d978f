"""Words handed to the host (r2s_fetch_begin / r2s_value_checks_begin): behind
long and short work, on several streams and threads, and when the work
launched meanwhile raises."""

import ctypes
import threading

import pytest
import torch

from r2splat_amd import _validation as check
from r2splat_amd import explicit, fused, workloads
from r2splat_amd.hip import _backend as be

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("n", [1, 2, 64])
@pytest.mark.parametrize("before", [0, 400])  # work ahead of the words: none, and several ms
def test_fetched_words_are_those_of_the_stream(device, n, before):
    x = torch.zeros(1 << 22, device=device)
    src = torch.empty(n, dtype=torch.int32, device=device)
    torch.cuda.synchronize(device)
    for k in range(3):
        for _ in range(before):
            x.add_(1.0)
        src.copy_(torch.arange(n, device=device, dtype=torch.int32) - 7 * k)
        words = be.fetch(src)
        src.fill_(99)  # launched behind the copy
        assert words.wait() == [i - 7 * k for i in range(n)]


def test_words_of_several_threads_and_streams(device):
    wrong = []

    def work(j):
        stream = torch.cuda.Stream(device)
        with torch.cuda.stream(stream):
            src = torch.empty(3, dtype=torch.int32, device=device)
            for k in range(50):
                src.fill_(100 * j + k)
                if be.fetch(src).wait() != [100 * j + k] * 3:
                    wrong.append((j, k))

    threads = [threading.Thread(target=work, args=(j,)) for j in range(4)]
    for t in threads:
        t.start()
    for t in threads:
        t.join()
    assert not wrong


def test_pending_checks_wait_when_the_work_raises(device):
    bad = torch.full((1000,), float("nan"), device=device)
    checks = check.ValueChecks()
    checks.finite("x", bad)
    with pytest.raises(KeyError):
        with checks.begin() as pending:
            raise KeyError("x")
    assert pending._words == []
    with pytest.raises(ValueError, match="x must contain only finite values"):
        pending.report()


def test_refused_adjoint_leaves_the_context_usable(device):
    sc = workloads.scene(300, 3, 40, 56, scale_range=(0.02, 0.08), seed=5, device=device)
    for recompute in (False, True):
        image, ctx = explicit.rasterize_fwd(*sc.params(), sc.viewmats, sc.Ks, sc.image_size, recompute=recompute)
        v = torch.ones_like(image)
        v[0, 3, 4] = float("inf")
        with pytest.raises(ValueError, match="v_image must contain only finite values"):
            explicit.rasterize_bwd(ctx, v)
        got = explicit.rasterize_bwd(ctx, torch.ones_like(image))
        _, again = explicit.rasterize_fwd(*sc.params(), sc.viewmats, sc.Ks, sc.image_size)
        assert torch.equal(got.means, explicit.rasterize_bwd(again, torch.ones_like(image)).means)


def test_forward_rendered_before_its_overflow_is_known(device):
    sc = workloads.scene(400, 2, 64, 64, scale_range=(0.05, 0.2), seed=9, device=device)
    args = (*sc.params(), sc.viewmats, sc.Ks, 64, 64, 1e-8, 3.0)
    expected, f = fused.forward(*args)
    image, g = fused.forward(*args, capacity=64)  # does not fit: rendered again with room
    assert f.n_isects == g.n_isects > 64
    assert torch.equal(image, expected)


def test_a_long_wait_keeps_another_calls_error(device):
    """The wait asks the runtime whether the stream has ended; an error that the
    thread has yet to read is not its own to clear."""
    path = next(line.split()[-1] for line in open("/proc/self/maps") if "libamdhip64" in line)
    hip = ctypes.CDLL(path)
    x = torch.zeros(1 << 24, device=device)
    src = torch.arange(2, device=device, dtype=torch.int32)
    torch.cuda.synchronize(device)
    for _ in range(600):  # some 20 ms: past the wait's spin
        x.add_(1.0)
    words = be.fetch(src)
    invalid = hip.hipSetDevice(10_000)
    assert invalid != 0 and hip.hipPeekAtLastError() == invalid
    try:
        assert words.wait() == [0, 1]
        assert hip.hipPeekAtLastError() == invalid
    finally:
        hip.hipGetLastError()
