"""Tile and level choices of the FP64 factorisation kernels.

The products behind the Cholesky factor, the triangular solve and the triangular
inverse run on 32, 64 or 128-wide tiles by the size of the launch, and the inverse
level by level over a recursion whose splits are ragged when n / 128 is no power of
two.  The sizes below sit on both sides of each choice (one leaf, two, odd counts of
leaves, and enough tiles for the 128-wide ones).
"""

import numpy as np
import pytest
import torch

from gpjax_amd import linalg

pytestmark = pytest.mark.gpu

EPS = np.finfo(np.float64).eps


def _spd(n):
    """exp(-|i - j| / 8) + I: condition number below 20, every entry known."""
    i = torch.arange(n, dtype=torch.float64, device="cuda")
    return torch.exp(-(i[:, None] - i[None, :]).abs() / 8) + torch.eye(n, dtype=torch.float64,
                                                                       device="cuda")


@pytest.mark.parametrize("n", [1, 127, 129, 384, 640, 897, 1153, 2049, 4225])
def test_factor_solve_and_inverse_residuals(n):
    A = _spd(n)
    L, logdet, info = linalg.cholesky_with_info(A)
    assert int(info) == 0
    # |L L^T - A| <= (n + 1) eps |L| |L|^T entrywise, each entry of |L| |L|^T at most
    # max A_ii = 2; twice that for the product formed here
    assert (L @ L.mT - A).abs().max() <= 2 * 2 * (n + 1) * EPS * 2
    assert torch.equal(L, torch.tril(L))
    sign, ref = np.linalg.slogdet(A.cpu().numpy())
    assert abs(float(logdet) - ref) <= 4 * n * EPS * max(1.0, abs(ref))
    # the products with L^-1: residuals within n eps ||L|| ||L^-1|| (condition < 5)
    B = torch.sin(torch.arange(3 * n, dtype=torch.float64, device="cuda")).reshape(n, 3)
    Y = linalg.solve_triangular(L, B)
    assert (L @ Y - B).abs().max() <= 8 * (n + 1) * EPS * 5 * B.abs().max()
    inv = linalg.inverse_from_cholesky(L)
    eye = torch.eye(n, dtype=torch.float64, device="cuda")
    assert (A @ inv - eye).abs().max() <= 8 * (n + 1) * EPS * 20
    assert torch.equal(inv, inv.mT.contiguous())
