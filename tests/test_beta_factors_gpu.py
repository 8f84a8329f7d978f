"""The native Beta line-integral factors against the reference's 160-digit
table and the torch forms, from tiny to huge exponents and one launch's edges."""

import json
from pathlib import Path

import pytest
import torch

from r2splat_amd._beta import beta_factors, beta_path_log_grad, beta_path_ratio

pytestmark = pytest.mark.gpu
ROWS = json.load(open(Path(__file__).parent / "golden" / "beta_path_factor.json"))["rows"]


@pytest.mark.parametrize("dtype", [torch.float32, torch.float64])
def test_native_factors_match_the_table(device, dtype):
    table = torch.tensor([[float(v) for v in row] for row in ROWS], dtype=torch.float64)
    gamma = table[:, 0].to(dtype)
    ratio, log_grad = beta_factors(gamma.to(device))
    exact = gamma.double() == table[:, 0]  # rows whose exponent the dtype holds
    # float64: at most 20 roundings of the recurrence; float32: one rounding
    tol = 4e-15 if dtype == torch.float64 else 1.2e-7
    for got, want in ((ratio, table[:, 1]), (log_grad, table[:, 2])):
        torch.testing.assert_close(got.cpu().double()[exact], want[exact], atol=0, rtol=tol)


@pytest.mark.parametrize("n", [1, 255, 256, 257, 5000])
def test_native_factors_match_the_torch_forms(device, n):
    g = torch.Generator().manual_seed(n)
    gamma = torch.exp(torch.rand(n, generator=g, dtype=torch.float64) * 12.0 - 6.0)
    ratio, log_grad = beta_factors(gamma.to(device))
    torch.testing.assert_close(ratio.cpu(), beta_path_ratio(gamma), atol=0, rtol=1e-13)
    torch.testing.assert_close(log_grad.cpu(), beta_path_log_grad(gamma), atol=0, rtol=1e-12)


def test_native_factors_outside_the_domain(device):
    gamma = torch.tensor([-0.75, -0.25, -1.3, -2.7, -7.45, float("nan"), float("inf")], dtype=torch.float64)
    ratio, log_grad = beta_factors(gamma.to(device))
    torch.testing.assert_close(ratio.cpu(), beta_path_ratio(gamma), atol=0, rtol=1e-12, equal_nan=True)
    torch.testing.assert_close(log_grad.cpu(), beta_path_log_grad(gamma), atol=1e-300, rtol=1e-10, equal_nan=True)
