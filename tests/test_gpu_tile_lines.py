"""The lines between the tile widths of the FP64 products.

A product runs on 32-wide tiles up to 24 tiles of 128 x 128, on 64-wide ones up to 512
and on 128-wide ones above, and every width sums k in the same order: the same columns
give the same bits on either side of a line.  A factorisation has products above the
second line from 8,192 rows on (the first trailing update), its level-by-level inverse
from 5,888 (23 x 23 tiles at the top).
"""

import numpy as np
import pytest
import torch

from gpjax_amd import linalg

pytestmark = pytest.mark.gpu

EPS = np.finfo(np.float64).eps


def _spd(n, device):
    """exp(-|i - j| / 8) + I: condition number below 20."""
    i = torch.arange(n, dtype=torch.float64, device=device)
    return torch.exp(-(i[:, None] - i[None, :]).abs() / 8) + torch.eye(n, dtype=torch.float64,
                                                                       device=device)


@pytest.mark.parametrize("n,tiles", [(128, (1, 24, 25, 512, 513)), (384, (1, 8, 9, 170, 171)),
                                     (600, (4, 5, 102, 103))])
def test_columns_keep_their_bits_across_the_lines(cuda, n, tiles):
    """L^-1 B for right-hand sides of `tiles` 128-column tiles (times n / 128 rows of
    them), all cut from one B: equal, bit for bit, and within n eps ||L|| ||L^-1||
    (condition < 5) of L Y = B."""
    L = torch.linalg.cholesky(_spd(n, "cpu")).to(cuda)
    rng = torch.Generator(device=cuda).manual_seed(n)
    B = torch.randn(n, 128 * max(tiles), generator=rng, dtype=torch.float64, device=cuda)
    wide = linalg.solve_triangular(L, B)
    assert (L @ wide - B).abs().max() <= 8 * (n + 1) * EPS * 5 * B.abs().max()
    for t in tiles:
        for m in (128 * t, 128 * t - 1):
            assert torch.equal(linalg.solve_triangular(L, B[:, :m]), wide[:, :m]), (t, m)


@pytest.mark.parametrize("n", [5900, 8200])
def test_factor_and_inverse_on_the_widest_tiles(cuda, n):
    """As the residuals of the smaller sizes: |L L^T - A| <= (n + 1) eps |L| |L|^T
    entrywise (entries at most 2, twice that for the product formed here), and
    A A^-1 - I within n eps times the condition."""
    A = _spd(n, cuda)
    L, logdet, info = linalg.cholesky_with_info(A)
    assert int(info) == 0
    assert torch.equal(L, torch.tril(L))
    assert (L @ L.mT - A).abs().max() <= 2 * 2 * (n + 1) * EPS * 2
    ref = 2.0 * torch.log(torch.diagonal(L)).sum()
    assert abs(float(logdet - ref)) <= 4 * n * EPS * max(1.0, abs(float(ref)))
    inv = linalg.inverse_from_cholesky(L)
    assert torch.equal(inv, inv.mT.contiguous())
    assert (A @ inv - torch.eye(n, dtype=torch.float64, device=cuda)).abs().max() <= \
        8 * (n + 1) * EPS * 20
