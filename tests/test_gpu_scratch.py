"""The scratch buffer in which dh_lra keeps K: its size, its return, and calls that
cannot have it, through the C ABI."""
import pytest

import darray_optimizer_amd as dh

pytestmark = pytest.mark.gpu


def problem(n, d, l, seed=0, labels=False):
    import torch
    g = torch.Generator(device="cuda").manual_seed(seed + n + d + l)
    X = 0.3 * torch.randn((n, d), dtype=torch.float64, device="cuda", generator=g)
    Om = torch.randn((l, n), dtype=torch.float64, device="cuda", generator=g)
    y = 0.5 + torch.rand(n, dtype=torch.float64, device="cuda", generator=g) if labels else None
    return X, Om, y


def solve(h, X, Om, q=1, y=None, prec=dh.DH_PREC_F64):
    import torch
    Q, W = torch.empty_like(Om), torch.empty_like(Om)
    assert h.lra(X, Om, 0.5 / X.shape[1], q, Q, W, y=y, prec=prec) == 0
    return Q, W


def test_scratch_is_reported_and_given_back(dev):
    """8 bytes per entry of K (rows in 64s, columns in 16s) after a solve, none after
    a trim, and the same solve again."""
    import torch
    X, Om, _ = problem(3001, 40, 24)
    dev.scratch_trim()
    assert dev.scratch_bytes() == 0
    a = solve(dev, X, Om)
    assert dev.scratch_bytes() == 8 * 3008 * 3008
    held = dev.workspace_bytes()
    dev.scratch_trim()
    assert dev.scratch_bytes() == 0 and dev.workspace_bytes() == held
    b = solve(dev, X, Om)
    assert torch.equal(a[0], b[0]) and torch.equal(a[1], b[1])
