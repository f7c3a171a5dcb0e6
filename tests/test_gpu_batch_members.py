"""A problem's result and gradient in a batch: the same bits whatever its company.

Every sum of a member is grouped by its padded size and input dimension alone, so one
GP gives the same floating-point numbers alone in its size group, among a few or among
hundreds (which run as pieces on several streams, with other launch shapes).
"""

import numpy as np
import pytest
import torch

import gpjax_amd as gpx

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("precision", ["fp64", "mixed"])
@pytest.mark.parametrize("n,d,counts", [(100, 7, (3, 600)), (128, 17, (5, 600)),
                                        (250, 7, (3, 500)), (600, 7, (2, 9, 160)),
                                        (1100, 6, (2, 24))])
def test_member_bits_do_not_depend_on_the_batch(cuda, monkeypatch, precision, n, d, counts):
    """Problem 0 alone, then first and last of batches of its padded size (sizes n and
    n - 1); nothing is tuned, since a tuned variant may order a sum differently."""
    monkeypatch.setattr(gpx.config, "mixed_check", "off")
    rng = np.random.default_rng(n + d)
    B = max(counts)
    Xs = [rng.uniform(0.0, 1.0, (n - p % 2, d)) for p in range(B)]
    ys = [np.sin(6 * X[:, 0]) + 0.1 * rng.standard_normal(len(X)) for X in Xs]
    ls = np.exp(rng.uniform(np.log(0.3), np.log(1.0), (B, d))) * np.sqrt(d)
    var, sd = rng.uniform(0.5, 2.0, B), rng.uniform(0.1, 0.3, B)

    def run(order):
        m = gpx.batched.BatchedConjugateMLL(
            [Xs[p] for p in order], [ys[p] for p in order], kernel="matern32",
            lengthscale=ls[order], variance=var[order], obs_stddev=sd[order],
            precision=precision, autotune=False)
        mll = m.mll()
        mll.sum().backward()
        return torch.cat([mll.detach().cpu()[:, None], m.lengthscale.value.grad.cpu(),
                          m.variance.value.grad.cpu()[:, None],
                          m.obs_stddev.value.grad.cpu()[:, None]], dim=1)

    alone = run([0])[0]
    assert torch.isfinite(alone).all()
    for count in counts:
        rest = list(range(1, count))
        assert torch.equal(run([0] + rest)[0], alone), count
        assert torch.equal(run(rest + [0])[-1], alone), count


@pytest.mark.parametrize("precision", ["fp64", "mixed"])
def test_tuner_times_what_runs(cuda, precision):
    """Variants that run the same kernels at a size are timed once and the plainer one is
    chosen: in float64 the gradient pass reads columns whatever the variant (d <= 32),
    and the solve of one leaf (n <= 128, d <= 16) evaluates Sigma itself, so a stored
    copy would be written for nothing.  The mixed path has all four."""
    rng = np.random.default_rng(3)
    sizes = [60, 100, 129, 500, 900]
    for d in (5, 18):
        Xs = [rng.uniform(0.0, 1.0, (n, d)) for n in sizes]
        ys = [np.sin(6 * X[:, 0]) for X in Xs]
        m = gpx.batched.BatchedConjugateMLL(Xs, ys, kernel="matern12", lengthscale=1.0,
                                            obs_stddev=0.2, precision=precision)
        assert [r["padded_size"] for r in m.tune_report] == [128, 256, 512, 1024]
        for r in m.tune_report:
            ms = r["ms"]
            assert all(t > 0 for t in ms.values())
            if precision == "mixed":
                assert len(set(ms.values())) > 1
                continue
            assert not r["transposed_pass"]
            assert ms["recomputed/transposed"] == ms["recomputed/columns"]
            assert ms["stored/transposed"] == ms["stored/columns"]
            if r["padded_size"] == 128 and d <= 16:
                assert not r["stored_sigma"]
                assert ms["stored/columns"] == ms["recomputed/columns"]
