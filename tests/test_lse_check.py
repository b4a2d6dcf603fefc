"""The LSE comparison of the GPU tests: rows without keys are checked, never skipped (CPU)."""

import numpy as np
import pytest

from tests.gpu_util import lse_max_err

NINF = -np.inf


def test_finite_rows_compared_and_empty_rows_accepted():
    ref = np.array([[1.0, NINF, 3.0]])
    out = np.zeros((1, 3, 2))
    out[0, 0] = 1.0
    out[0, 2] = 2.0
    assert lse_max_err(np.array([[1.25, NINF, 3.0]]), ref, out) == 0.25


@pytest.mark.parametrize("bad", [np.nan, 0.0, 5.0])
def test_empty_row_must_be_neg_inf(bad):
    with pytest.raises(AssertionError):
        lse_max_err(np.array([[1.0, bad]]), np.array([[1.0, NINF]]))


def test_nan_in_a_finite_row_fails():
    with pytest.raises(AssertionError):
        lse_max_err(np.array([[np.nan, 2.0]]), np.array([[1.0, 2.0]]))


def test_empty_row_output_must_be_zero():
    out = np.zeros((1, 2, 4))
    out[0, 1, 3] = 1e-3
    with pytest.raises(AssertionError):
        lse_max_err(np.array([[1.0, NINF]]), np.array([[1.0, NINF]]), out)


def test_finish_lse_keeps_graph_and_tangent(monkeypatch):
    """The smoothing correction of an LSE stays differentiable in Q, in reverse and in forward mode: neither takes the
    kernel that writes lse in place."""
    import torch
    import torch.autograd.forward_ad as fwd

    from telefuser_amd import _lib
    from telefuser_amd import sageattn2 as sa

    def no_kernel():
        raise AssertionError("the kernel was called")

    monkeypatch.setattr(_lib, "load", no_kernel)
    g = torch.Generator().manual_seed(1)
    q, t = (torch.randn((2, 5, 4, 64), generator=g) for _ in range(2))  # NHD, grouped heads
    km, lse = torch.randn((2, 2, 64), generator=g), torch.randn((2, 4, 5), generator=g)
    want = torch.einsum("blhd,bhd->bhl", t, km.repeat_interleave(2, dim=1)) * 0.125
    with fwd.dual_level():
        out = fwd.unpack_dual(sa._finish_lse(lse.clone(), fwd.make_dual(q, t), km, "NHD", 0.125))
        torch.testing.assert_close(out.tangent, want)
    qr = q.clone().requires_grad_()
    got = sa._finish_lse(lse.clone(), qr, km, "NHD", 0.125)
    torch.testing.assert_close(got.detach(), out.primal)
    (grad,) = torch.autograd.grad(got.sum(), qr)
    torch.testing.assert_close(grad, (km.repeat_interleave(2, dim=1) * 0.125)[:, None].expand_as(q))
